// Minimum-image vectors and hop neighbour lists on gfx950.
//
//   pycd_min_image_vectors  <- Neighbors.get_pairwise_min_image_vector_data
//                              (PyCD/core.py:571-594): N x N x 3 vectors
//                              pos[j] - pos[i] under the minimum image
//   pycd_hop_neighbors      <- Neighbors.hop_neighbor_sites /
//                              generate_neighbor_list (PyCD/core.py:485-668):
//                              per centre and shell, the targets with
//                              lo < |r| <= hi in ascending target order
//
// The minimum image follows PyCD/core.py:304-361: fractional coordinates,
// round-half-even base offset on periodic axes, then the 26 neighbouring
// offsets in (dx, dy, dz) loop order, a candidate replacing the best only if
// strictly shorter.
#include "common.hpp"
#include "ewald_common.hpp"

namespace pycd {

__device__ inline double mic_vec(double dx, double dy, double dz,
                                 const MicGeometry& g, double* v) {
  double f0 = dx * g.inv[0] + dy * g.inv[3] + dz * g.inv[6];
  double f1 = dx * g.inv[1] + dy * g.inv[4] + dz * g.inv[7];
  double f2 = dx * g.inv[2] + dy * g.inv[5] + dz * g.inv[8];
  if (g.pbc[0]) f0 -= rint(f0);
  if (g.pbc[1]) f1 -= rint(f1);
  if (g.pbc[2]) f2 -= rint(f2);
  double bx = f0 * g.cell[0] + f1 * g.cell[3] + f2 * g.cell[6];
  double by = f0 * g.cell[1] + f1 * g.cell[4] + f2 * g.cell[7];
  double bz = f0 * g.cell[2] + f1 * g.cell[5] + f2 * g.cell[8];
  double best = bx * bx + by * by + bz * bz;
  double vx = bx, vy = by, vz = bz;
  for (int m = 0; m < g.n_delta; ++m) {
    const double cx = bx + g.dS[m][0];
    const double cy = by + g.dS[m][1];
    const double cz = bz + g.dS[m][2];
    const double r2 = cx * cx + cy * cy + cz * cz;
    if (r2 < best) {
      best = r2;
      vx = cx;
      vy = cy;
      vz = cz;
    }
  }
  v[0] = vx;
  v[1] = vy;
  v[2] = vz;
  return sqrt(best);
}

__global__ void __launch_bounds__(256)
min_image_kernel(const double* __restrict__ pos, int64_t n, MicGeometry g,
                 double* __restrict__ out) {
  const int64_t total = n * n;
  for (int64_t idx = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
       idx < total; idx += int64_t(gridDim.x) * blockDim.x) {
    const int64_t i = idx / n, j = idx - i * n;
    double v[3];
    mic_vec(pos[3 * j] - pos[3 * i], pos[3 * j + 1] - pos[3 * i + 1],
            pos[3 * j + 2] - pos[3 * i + 2], g, v);
    out[3 * idx] = v[0];
    out[3 * idx + 1] = v[1];
    out[3 * idx + 2] = v[2];
  }
}

constexpr int kMaxShells = 16;

struct ShellWindows {
  double lo[kMaxShells];
  double hi[kMaxShells];
  int n;
  // |f_k| above far[k] (f the wrapped fractional difference): every image
  // is beyond the widest window
  double far[3];
};

// One wavefront per kC centres; lanes sweep the targets 64 at a time in
// ascending order, and a ballot per shell gives each hit its rank.
//
// Few centres: bound by the chain of a sweep's steps, so the positions are
// loaded one step ahead and their indices two.  Many: by FP64 instructions
// per pair.  A pair whose wrapped fractional difference exceeds `far` on an
// axis is beyond every window: |f_k| <= |d| times the length of column k of
// S^-1, no image has a smaller |f_k| than the wrapped one, and the margin of
// `far` (1e-6) is above the rounding of f for sites up to 1e9 cells away.
// Only the others form the minimum image (9 products for f, 9 for the
// vector, 7 for each of 12 images); 64 targets that all fail cost their
// fractional coordinates (9 products, shared by the wavefront's centres)
// and per centre and axis a subtraction, a wrap and a comparison.  Shells
// to 3.0 A, 6144 centres x 6144 targets: 259 us with a minimum image per
// pair, 73 so; 768 x 768: 26 and 21 us.  (With the fractional coordinates
// read from an array that a kernel ahead filled, the second launch cost a
// call 30-40 us up to 6144 sites.)
template <int kC>
__global__ void __launch_bounds__(256)
hop_neighbor_kernel(const double* __restrict__ pos,
                    const int64_t* __restrict__ centers, int64_t n_centers,
                    const int64_t* __restrict__ targets, int64_t n_targets,
                    MicGeometry g, ShellWindows w, int max_per,
                    int32_t* __restrict__ count, int32_t* __restrict__ index,
                    double* __restrict__ vec) {
  const int lane = threadIdx.x & 63;
  const int64_t c0 =
      (int64_t(blockIdx.x) * 4 +
       __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * kC;
  if (c0 >= n_centers) return;
  double px[kC], py[kC], pz[kC], fc[kC][3];
  int running[kC][kMaxShells];
#pragma unroll
  for (int u = 0; u < kC; ++u) {
    // (a missing centre repeats the last one and stores nothing)
    const int64_t ci = centers[c0 + u < n_centers ? c0 + u : n_centers - 1];
    px[u] = pos[3 * ci];
    py[u] = pos[3 * ci + 1];
    pz[u] = pos[3 * ci + 2];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      fc[u][k] = px[u] * g.inv[k] + py[u] * g.inv[3 + k] + pz[u] * g.inv[6 + k];
#pragma unroll
    for (int s = 0; s < kMaxShells; ++s) running[u][s] = 0;
  }
  const unsigned long long below =
      lane == 0 ? 0ull : (~0ull >> (64 - lane));
  // axes that do not wrap subtract rint(f) times 0
  const double wrap[3] = {g.pbc[0] ? 1.0 : 0.0, g.pbc[1] ? 1.0 : 0.0,
                          g.pbc[2] ? 1.0 : 0.0};
  // lanes past the last target repeat the first and report nothing
  double qn[3];
  const int64_t t0 = targets[lane < n_targets ? lane : 0];
#pragma unroll
  for (int k = 0; k < 3; ++k) qn[k] = pos[3 * t0 + k];
  int64_t tn = targets[lane + 64 < n_targets ? lane + 64 : 0];
  for (int64_t j0 = 0; j0 < n_targets; j0 += 64) {
    const int64_t j = j0 + lane;
    const bool real = j < n_targets;
    double q[3], f[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      q[k] = qn[k];
      qn[k] = pos[3 * tn + k];
    }
    tn = targets[j + 128 < n_targets ? j + 128 : 0];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      f[k] = q[0] * g.inv[k] + q[1] * g.inv[3 + k] + q[2] * g.inv[6 + k];
#pragma unroll
    for (int u = 0; u < kC; ++u) {
      bool near = real;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const double d = f[k] - fc[u][k];
        near = near && !(fabs(fma(-wrap[k], rint(d), d)) > w.far[k]);
      }
      if (__ballot(near) == 0ull) continue;
      double v[3] = {0.0, 0.0, 0.0};
      double r = -1.0;
      if (near)
        r = mic_vec(q[0] - px[u], q[1] - py[u], q[2] - pz[u], g, v);
#pragma unroll
      for (int s = 0; s < kMaxShells; ++s) {
        if (s >= w.n) break;
        const bool in = near && w.lo[s] < r && r <= w.hi[s];
        const unsigned long long mask = __ballot(in);
        if (in) {
          const int rank = running[u][s] + __popcll(mask & below);
          if (rank < max_per && c0 + u < n_centers) {
            const int64_t o = ((c0 + u) * w.n + s) * max_per + rank;
            index[o] = int32_t(j);
            vec[3 * o] = v[0];
            vec[3 * o + 1] = v[1];
            vec[3 * o + 2] = v[2];
          }
        }
        running[u][s] += __popcll(mask);
      }
    }
  }
#pragma unroll
  for (int u = 0; u < kC; ++u)
#pragma unroll
    for (int s = 0; s < kMaxShells; ++s) {
      if (s >= w.n || c0 + u >= n_centers) break;
      const int64_t row = (c0 + u) * w.n + s;
      if (lane == 0) count[row] = running[u][s];
      // the room past the shell's entries: the block is a kept one
      for (int r = running[u][s] + lane; r < max_per; r += 64) {
        const int64_t o = row * max_per + r;
        index[o] = 0;
        vec[3 * o] = 0.0;
        vec[3 * o + 1] = 0.0;
        vec[3 * o + 2] = 0.0;
      }
    }
}

}  // namespace pycd

using namespace pycd;

extern "C" int pycd_min_image_vectors(pycd_ctx* ctx, const double* pos,
                                      int64_t n, const double cell[9],
                                      const int32_t pbc[3], double* out) {
  if (!ctx) return PYCD_ERR_ARG;
  if (!pos || !cell || !pbc || !out || n <= 0 || n > (int64_t(1) << 17))
    return fail(ctx, PYCD_ERR_ARG, "bad minimum-image arguments");
  DeviceGuard guard(ctx->device);
  hipStream_t st = ctx->stream;
  MicGeometry g;
  fill_mic_geometry(cell, pbc, g);
  WorkBuf<double> dpos, dout;
  PYCD_HIP(ctx, dpos.alloc(ctx, size_t(n) * 3));
  PYCD_HIP(ctx, upload(dpos.ptr, pos, size_t(n) * 3, st));
  double* o = out;
  const bool out_dev = is_device_ptr(out);
  if (!out_dev) {
    PYCD_HIP(ctx, dout.alloc(ctx, size_t(n) * n * 3));
    o = dout.ptr;
  }
  const int64_t total = n * n;
  const int blocks = int(std::min<int64_t>((total + 255) / 256, 1 << 20));
  min_image_kernel<<<blocks, 256, 0, st>>>(dpos.ptr, n, g, o);
  PYCD_HIP(ctx, hipGetLastError());
  if (!out_dev)
    PYCD_HIP(ctx, hipMemcpyAsync(out, o, 8 * 3 * size_t(total),
                                 hipMemcpyDeviceToHost, st));
  PYCD_HIP(ctx, hipStreamSynchronize(st));
  return PYCD_OK;
}

extern "C" int pycd_hop_neighbors(pycd_ctx* ctx, const double* pos, int64_t n,
                                  const int64_t* centers, int64_t n_centers,
                                  const int64_t* targets, int64_t n_targets,
                                  const double cell[9], const int32_t pbc[3],
                                  const double* lo, const double* hi,
                                  int32_t n_shells, int32_t max_per_shell,
                                  int32_t* count, int32_t* index,
                                  double* vec) {
  if (!ctx) return PYCD_ERR_ARG;
  if (!pos || !centers || !targets || !cell || !pbc || !lo || !hi || !count ||
      !index || !vec || n <= 0 || n_centers <= 0 || n_targets <= 0 ||
      n_shells <= 0 || n_shells > kMaxShells || max_per_shell <= 0 ||
      n_centers > (int64_t(1) << 24) || n_targets > (int64_t(1) << 24))
    return fail(ctx, PYCD_ERR_ARG, "bad neighbour-list arguments");
  for (int64_t k = 0; k < n_centers; ++k)
    if (centers[k] < 0 || centers[k] >= n)
      return fail(ctx, PYCD_ERR_ARG, "centre index out of range");
  for (int64_t k = 0; k < n_targets; ++k)
    if (targets[k] < 0 || targets[k] >= n)
      return fail(ctx, PYCD_ERR_ARG, "target index out of range");
  DeviceGuard guard(ctx->device);
  hipStream_t st = ctx->stream;
  MicGeometry g;
  fill_mic_geometry(cell, pbc, g);
  ShellWindows w;
  w.n = n_shells;
  for (int s = 0; s < kMaxShells; ++s) {
    w.lo[s] = s < n_shells ? lo[s] : 0.0;
    w.hi[s] = s < n_shells ? hi[s] : -1.0;
  }
  double reach = 0.0;
  for (int s = 0; s < n_shells; ++s)
    if (!(hi[s] <= reach)) reach = hi[s];
  for (int k = 0; k < 3; ++k) {
    const double* c = g.inv + k;
    w.far[k] = reach * std::sqrt(c[0] * c[0] + c[3] * c[3] + c[6] * c[6]) *
                   (1.0 + 1e-9) + 1e-6;
  }
  const size_t nout = size_t(n_centers) * n_shells * max_per_shell;
  WorkBuf<double> dpos, dvec;
  WorkBuf<int64_t> dc, dt;
  WorkBuf<int32_t> dcount, dindex;
  PYCD_HIP(ctx, dpos.alloc(ctx, size_t(n) * 3));
  PYCD_HIP(ctx, dc.alloc(ctx, n_centers));
  PYCD_HIP(ctx, dt.alloc(ctx, n_targets));
  PYCD_HIP(ctx, dcount.alloc(ctx, size_t(n_centers) * n_shells));
  PYCD_HIP(ctx, dindex.alloc(ctx, nout));
  PYCD_HIP(ctx, dvec.alloc(ctx, nout * 3));
  PYCD_HIP(ctx, upload(dpos.ptr, pos, size_t(n) * 3, st));
  PYCD_HIP(ctx, hipMemcpyAsync(dc.ptr, centers, 8 * n_centers,
                               hipMemcpyHostToDevice, st));
  PYCD_HIP(ctx, hipMemcpyAsync(dt.ptr, targets, 8 * n_targets,
                               hipMemcpyHostToDevice, st));
  // More centres per wavefront share more of each pair's work and leave
  // fewer wavefronts: a call (as many targets, two shells of 4) with 1, 2, 4
  // each takes 170, 177, 203 us at 4116 centres, 195, 198, 228 at 5376, 230,
  // 228, 257 at 6144, 323, 294, 322 at 8748, 469, 392, 405 at 12000, 661, 533,
  // 502 at 15972, 1104, 790, 740 at 22464.
  const auto launch = [&](auto kernel, int per_wave) {
    const int64_t per_block = 4 * per_wave;
    kernel<<<unsigned((n_centers + per_block - 1) / per_block), 256, 0, st>>>(
        dpos.ptr, dc.ptr, n_centers, dt.ptr, n_targets, g, w, max_per_shell,
        dcount.ptr, dindex.ptr, dvec.ptr);
  };
  if (n_centers < 6144)
    launch(hop_neighbor_kernel<1>, 1);
  else if (n_centers < 13824)
    launch(hop_neighbor_kernel<2>, 2);
  else
    launch(hop_neighbor_kernel<4>, 4);
  PYCD_HIP(ctx, hipGetLastError());
  PYCD_HIP(ctx, hipMemcpyAsync(count, dcount.ptr,
                               4 * size_t(n_centers) * n_shells,
                               hipMemcpyDeviceToHost, st));
  PYCD_HIP(ctx, hipMemcpyAsync(index, dindex.ptr, 4 * nout,
                               hipMemcpyDeviceToHost, st));
  PYCD_HIP(ctx, hipMemcpyAsync(vec, dvec.ptr, 8 * 3 * nout,
                               hipMemcpyDeviceToHost, st));
  PYCD_HIP(ctx, hipStreamSynchronize(st));
  for (size_t k = 0; k < size_t(n_centers) * n_shells; ++k)
    if (count[k] > max_per_shell)
      return fail(ctx, PYCD_ERR_ARG,
                  "a shell holds %d targets (> max_per_shell %d); counts are "
                  "returned",
                  count[k], max_per_shell);
  return PYCD_OK;
}
