// Live-frame maps and projective frame-to-model ICP.
//
// Reference: include/image/sensor/rgbdImage.cu (creatPointCloudKernel :22-38,
// vertextoNormal :126-145), include/image/pyramid/pyramid.cu (downsampling
// :48-82), include/solver/gnSolver/gnSolver.cu (buildNLSKernel :25-196,
// solve :317-438).
//
// Per iteration the reduction kernel evaluates one Gauss-Newton linearisation
// per pixel and reduces the 30 sums (21 of J J^T, 6 of J r, counts) with a
// wavefront shuffle tree plus an LDS stage into one record per workgroup; the
// session's last workgroup adds the records in FP64 in a fixed order, solves
// the damped 6x6 system with an FP64 LDL^T and composes the SE(3) increment, so
// an iteration is one launch and a frame's iterations run back to back without
// a host round trip.
#include "dm_device.h"
#include "dm_solve.h"

namespace dm {

__device__ __forceinline__ Intr level_intr(const DmView &v, int l) {
  const float s = (float)(1 << l);
  return Intr{v.rows >> l, v.cols >> l, v.fx / s, v.fy / s, v.cx / s, v.cy / s};
}

__device__ __forceinline__ float intensity_rgb(const uint8_t *rgb, int idx) {
  if (!rgb) return 0.f;
  return (0.2126f * (float)rgb[3 * idx] + 0.7152f * (float)rgb[3 * idx + 1] + 0.0722f * (float)rgb[3 * idx + 2]) *
         (1.0f / 255.0f);
}

// depth of level-l pixel j, taken from the level-0 frame at (2^l u, 2^l v)
__device__ __forceinline__ float level_depth(const DmView &v, int l, int j, int cols_l) {
  const int vv = j / cols_l, uu = j - vv * cols_l;
  const float *d = v.depth_track ? v.depth_track : v.depth;
  return d[(size_t)(vv << l) * v.cols + (uu << l)];
}

// Vertex of level-l pixel j.  D: evaluated in FP64 and rounded to float, so
// the live-frame maps equal the FP64 oracle's (depth <= 0 gives (0,0,0)).
__device__ __forceinline__ f3 level_vertex(const DmView &v, int l, int j, const Intr &s) {
  const float d = level_depth(v, l, j, s.cols);
  if (!(d > 0.0f)) return mk(0.f, 0.f, 0.f);
  const int vv = j / s.cols, uu = j - vv * s.cols;
  const double dd = (double)d;
  return mk((float)((((double)uu - (double)s.cx) * dd) / (double)s.fx),
            (float)((((double)vv - (double)s.cy) * dd) / (double)s.fy), d);
}

// Source maps of all pyramid levels straight from the level-0 depth:
// vertex (creatPointCloudKernel), intensity, and the normal of
// vertextoNormal (K: cross(V[i+2]-V[i-2], V[i+W]-V[i-W]) with out-of-range
// neighbours replaced by the pixel itself; D: NaN when a neighbour has no
// depth, evaluated in FP64).  D: level l is the true (rows>>l) x (cols>>l)
// nearest subsample.
__global__ __launch_bounds__(256) void k_source_maps(const DmView *__restrict__ views, const int *__restrict__ active) {
  const int slot_ = active[blockIdx.y];
  if (slot_ < 0) return;
  const DmView &v = views[slot_];
  const int P0 = v.rows * v.cols;
  const int P1 = (v.rows >> 1) * (v.cols >> 1);
  const int P2 = (v.rows >> 2) * (v.cols >> 2);
  int t = blockIdx.x * 256 + threadIdx.x;
  int l;
  if (t < P0) l = 0;
  else if (t < P0 + P1) { l = 1; t -= P0; }
  else if (t < P0 + P1 + P2) { l = 2; t -= P0 + P1; }
  else return;
  const Intr s = level_intr(v, l);
  const int size = s.rows * s.cols;
  const f3 c = level_vertex(v, l, t, s);
  const int vv = t / s.cols, uu = t - vv * s.cols;
  const float inten = intensity_rgb(v.rgb, (vv << l) * v.cols + (uu << l));
  v.svert[l][t] = make_float4(c.x, c.y, c.z, inten);
  const int li = t - 2 < 0 ? t : t - 2;
  const int ri = t + 2 >= size ? t : t + 2;
  const int ui = t - s.cols <= 0 ? t : t - s.cols;
  const int di = t + s.cols >= size ? t : t + s.cols;
  const f3 L = level_vertex(v, l, li, s), R = level_vertex(v, l, ri, s), U = level_vertex(v, l, ui, s),
           D = level_vertex(v, l, di, s);
  float4 n;
  if (L.z == 0.f || R.z == 0.f || U.z == 0.f || D.z == 0.f || c.z == 0.f) {
    const float qn = __int_as_float(0x7fc00000);
    n = make_float4(qn, qn, qn, 0.f);
  } else {
    const double ax = (double)R.x - (double)L.x, ay = (double)R.y - (double)L.y, az = (double)R.z - (double)L.z;
    const double bx = (double)D.x - (double)U.x, by = (double)D.y - (double)U.y, bz = (double)D.z - (double)U.z;
    const double cx = ay * bz - az * by, cy = az * bx - ax * bz, cz = ax * by - ay * bx;
    const double nn = sqrt(cx * cx + cy * cy + cz * cz);
    n = make_float4((float)(cx / nn), (float)(cy / nn), (float)(cz / nn), 0.f);
  }
  v.snorm[l][t] = n;
}

constexpr int kVals = 30;

// Association and gates of one pixel (buildNLSKernel, gnSolver.cu:55-195).
// K: Project() association, the |cos| > cos(pi/10) normal gate, r =
// (p - q).n, J = [p x n; n].  D: source normal rotated by Tinc, pixel bounds
// check, |p - q| <= dist_max, depth gate [icp_dmin, icp_dmax].  The
// transform, projection and gates are in FP64 (the pixel choice and the
// inclusion decisions follow the FP64 geometry); residual and Jacobian are
// FP32.
//
// The pixels of a thread go through the three rounds of loads (source point and
// normal; model point and normal; the model intensity's neighbours) side by
// side, every load unconditional at a safe index: taken one pixel after the
// other, each load behind the test of the one before, an iteration of a coarse
// level was 12 rounds of memory latency (16 sessions at level 0 74 -> 58 us; one
// session's iterations at icp_record).  The rest of an iteration is a chain too:
// 7000 of 34000 cycles the four pixels' arithmetic on few wavefronts, 3000 the
// tickets, 3500 the records, 9000 the step.  One pixel per thread in workgroups
// of 1024 took as long (the same wavefronts' work on the same compute unit).
constexpr int kIcpPer = kIcpPix / 256;  // pixels per thread
typedef float f32x4 __attribute__((ext_vector_type(4)));
struct IcpPixel {
  double px, py, pz;    // transformed source point
  f32x4 Q, NT;          // model point (w: intensity) and normal
  f3 N;                 // source normal
  float vw;             // source intensity
  float xp, xm, yp, ym; // model intensity beside the associated pixel
  bool ok, inner;       // associated; with the four neighbours inside the image
};
__device__ __forceinline__ double uniform_f64(double x) {
  return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(x)),
                          __builtin_amdgcn_readfirstlane(__double2loint(x)));
}
struct IcpPose { double m[12]; };
__device__ __forceinline__ IcpPose icp_pose(const DmView &v) {
  double m[12];
#pragma unroll
  for (int k = 0; k < 12; ++k) m[k] = ldg(v.posed + PD_TINC + k);
  IcpPose T;
#pragma unroll
  for (int k = 0; k < 12; ++k) T.m[k] = uniform_f64(m[k]);
  return T;
}
__device__ __forceinline__ bool bad3(f32x4 n) {
  return !(fabsf(n.x) <= 3.4e38f) || !(fabsf(n.y) <= 3.4e38f) || !(fabsf(n.z) <= 3.4e38f) ||
         (n.x == 0.f && n.y == 0.f && n.z == 0.f);
}
__device__ __forceinline__ void icp_pixels(const DmView &v, int level, const Intr &s, int P, IcpPose &T,
                                           IcpPixel (&a)[kIcpPer]) {
  const f32x4 *sv = reinterpret_cast<const f32x4 *>(v.svert[level]), *sn = reinterpret_cast<const f32x4 *>(v.snorm[level]);
  const f32x4 *tv = reinterpret_cast<const f32x4 *>(v.tvert[level]), *tn = reinterpret_cast<const f32x4 *>(v.tnorm[level]);
  f32x4 V[kIcpPer], N[kIcpPer];
#pragma unroll
  for (int q = 0; q < kIcpPer; ++q) {
    const int i = min((int)blockIdx.x * kIcpPix + q * 256 + (int)threadIdx.x, P - 1);
    V[q] = ldg(sv + i);
    N[q] = ldg(sn + i);
  }
  T = icp_pose(v);
  const double *Td = T.m;
  int j[kIcpPer];
#pragma unroll
  for (int q = 0; q < kIcpPer; ++q) {
    IcpPixel &x = a[q];
    x.ok = (int)blockIdx.x * kIcpPix + q * 256 + (int)threadIdx.x < P && V[q].z >= v.icp_dmin &&
           V[q].z <= v.icp_dmax && !bad3(N[q]);
    const double X = V[q].x, Y = V[q].y, Z = V[q].z;
    x.px = Td[0] * X + Td[1] * Y + Td[2] * Z + Td[3];
    x.py = Td[4] * X + Td[5] * Y + Td[6] * Z + Td[7];
    x.pz = Td[8] * X + Td[9] * Y + Td[10] * Z + Td[11];
    const int pu = to_i32d(round(((double)s.fx * x.px) / x.pz + (double)s.cx));
    const int pv = to_i32d(round(((double)s.fy * x.py) / x.pz + (double)s.cy));
    x.ok = x.ok && !(pu < 0 || pv < 0 || pu >= s.cols || pv >= s.rows);
    x.inner = x.ok && pu >= 1 && pv >= 1 && pu < s.cols - 1 && pv < s.rows - 1;
    x.N = mk(N[q].x, N[q].y, N[q].z);
    x.vw = V[q].w;
    j[q] = x.ok ? pv * s.cols + pu : 0;
  }
#pragma unroll
  for (int q = 0; q < kIcpPer; ++q) {
    a[q].Q = ldg(tv + j[q]);
    a[q].NT = ldg(tn + j[q]);
  }
  if (v.w_photo > 0.f) {
#pragma unroll
    for (int q = 0; q < kIcpPer; ++q) {
      const int dx = a[q].inner ? 1 : 0, dy = a[q].inner ? s.cols : 0;
      a[q].xp = ldg((const float *)(tv + j[q] + dx) + 3);
      a[q].xm = ldg((const float *)(tv + j[q] - dx) + 3);
      a[q].yp = ldg((const float *)(tv + j[q] + dy) + 3);
      a[q].ym = ldg((const float *)(tv + j[q] - dy) + 3);
    }
  }
}
// The gates; p: the transformed source point, pq: p - q.
__device__ __forceinline__ bool icp_gate(const DmView &v, const IcpPose &T, const IcpPixel &x, f3 &p, f3 &pq) {
  const double *Td = T.m;
  const double X = x.N.x, Y = x.N.y, Z = x.N.z;
  const double nrx = Td[0] * X + Td[1] * Y + Td[2] * Z;
  const double nry = Td[4] * X + Td[5] * Y + Td[6] * Z;
  const double nrz = Td[8] * X + Td[9] * Y + Td[10] * Z;
  const double ct = (double)x.NT.x * nrx + (double)x.NT.y * nry + (double)x.NT.z * nrz;
  const double dqx = x.px - (double)x.Q.x, dqy = x.py - (double)x.Q.y, dqz = x.pz - (double)x.Q.z;
  p = mk((float)x.px, (float)x.py, (float)x.pz);
  pq = mk((float)dqx, (float)dqy, (float)dqz);
  // sqrt(d2) <= dist_max, from the squares unless they are equal to 1e-12
  const double d2 = dqx * dqx + dqy * dqy + dqz * dqz, dm = (double)v.dist_max, m2 = dm * dm;
  bool near = dm >= 0.0 && d2 < m2;
  if (!(fabs(d2 - m2) > 1e-12 * m2)) near = sqrt(d2) <= dm;
  return x.ok && x.Q.z >= v.icp_dmin && x.Q.z <= v.icp_dmax && !bad3(x.NT) && fabs(ct) > 0.95105651629515357 && near;
}

// Per-pixel terms of one Gauss-Newton linearisation
// accumulated into vals (upper JtJ 21, Jtr 6, geometric count, r^2,
// photometric count); the photometric term adds w_photo Jp Jp^T and
// w_photo Jp rp.
__device__ __forceinline__ void icp_terms(const DmView &v, const Intr &s, const IcpPose &T, const IcpPixel &x,
                                          float *vals) {
  f3 p, pq;
  if (!icp_gate(v, T, x, p, pq)) return;
  const f3 n = mk(x.NT.x, x.NT.y, x.NT.z);
  float pvl[kVals];
  const float r = dot(pq, n);
  const f3 c = cross(p, n);
  const float J[6] = {c.x, c.y, c.z, n.x, n.y, n.z};
  int k = 0;
#pragma unroll
  for (int a = 0; a < 6; ++a)
#pragma unroll
    for (int b = a; b < 6; ++b) pvl[k++] = J[a] * J[b];
#pragma unroll
  for (int a = 0; a < 6; ++a) pvl[21 + a] = J[a] * r;
  pvl[27] = 1.f;
  pvl[28] = r * r;
  pvl[29] = 0.f;
  if (v.w_photo > 0.f && x.inner) {
    const float gx = (x.xp - x.xm) * 0.5f;
    const float gy = (x.yp - x.ym) * 0.5f;
    const float rp = x.Q.w - x.vw;
    const float iz = 1.0f / p.z;
    const f3 G = mk(gx * s.fx * iz, gy * s.fy * iz, -(gx * s.fx * p.x + gy * s.fy * p.y) * iz * iz);
    const f3 cg = cross(p, G);
    const float Jp[6] = {cg.x, cg.y, cg.z, G.x, G.y, G.z};
    const float wp = v.w_photo;
    int kk = 0;
#pragma unroll
    for (int a = 0; a < 6; ++a)
#pragma unroll
      for (int b = a; b < 6; ++b) { pvl[kk] = pvl[kk] + wp * Jp[a] * Jp[b]; ++kk; }
#pragma unroll
    for (int a = 0; a < 6; ++a) pvl[21 + a] = pvl[21 + a] + wp * Jp[a] * rp;
    pvl[29] = 1.f;
  }
#pragma unroll
  for (int q = 0; q < kVals; ++q) vals[q] = vals[q] + pvl[q];
}

// The feature row of one pixel for the matrix-core reduction: geometric
// [J, r, 1] in columns 0-7 and photometric sqrt(w_photo) [Jp, rp] with a 1 in
// columns 8-15 (zeros where a term does not apply).  F^T F summed over the
// pixels holds J^T J and J^T r of both terms, r^2 and both counts.
__device__ __forceinline__ void icp_features(const DmView &v, const Intr &s, const IcpPose &T, const IcpPixel &x,
                                             float swp, float *f) {
#pragma unroll
  for (int k = 0; k < 16; ++k) f[k] = 0.f;
  f3 p, pq;
  if (!icp_gate(v, T, x, p, pq)) return;
  const f3 n = mk(x.NT.x, x.NT.y, x.NT.z);
  const float r = dot(pq, n);
  const f3 c = cross(p, n);
  f[0] = c.x; f[1] = c.y; f[2] = c.z; f[3] = n.x; f[4] = n.y; f[5] = n.z; f[6] = r; f[7] = 1.f;
  if (v.w_photo > 0.f && x.inner) {
    const float gx = (x.xp - x.xm) * 0.5f;
    const float gy = (x.yp - x.ym) * 0.5f;
    const float rp = x.Q.w - x.vw;
    const float iz = 1.0f / p.z;
    const f3 G = mk(gx * s.fx * iz, gy * s.fy * iz, -(gx * s.fx * p.x + gy * s.fy * p.y) * iz * iz);
    const f3 cg = cross(p, G);
    f[8] = swp * cg.x; f[9] = swp * cg.y; f[10] = swp * cg.z;
    f[11] = swp * G.x; f[12] = swp * G.y; f[13] = swp * G.z;
    f[14] = swp * rp; f[15] = 1.f;
  }
}

// ---- the Gauss-Newton step on the device
// Value of lane `l` (uniform) in every lane.
__device__ __forceinline__ double lane_f64(double x, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), l),
                          __builtin_amdgcn_readlane(__double2loint(x), l));
}
// Largest value of lanes 0..31, ignoring NaN.
__device__ __forceinline__ double max_f64(double a, double b) { return b > a || a != a ? b : a; }
__device__ __forceinline__ double half_max(double x) {
  x = max_f64(x, dpp_f64<0xb1>(x));
  x = max_f64(x, dpp_f64<0x4e>(x));
  x = max_f64(x, dpp_f64<0x141>(x));
  x = max_f64(x, dpp_f64<0x140>(x));
  return max_f64(x, __shfl_xor(x, 16, 64));
}

// Scratch of the step in LDS.
struct IcpStepLds {
  double part[32][32];    // sums of 8 leaves each, by value
  double pd[PD_COUNT];    // the session's pose block
  double m[16], t[16];    // matrices handed between lanes
};

// A record value: written by other workgroups of the same launch, so it is
// read past this XCD's caches.
__device__ __forceinline__ float record_value(const float *p) {
  return __hip_atomic_load((const __attribute__((address_space(1))) float *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The damped Gauss-Newton step of one session, by one workgroup of 256
// threads once every record of the linearisation is stored.
// Sum: leaf t of 256 adds records t, t + 256, ... in order, and the leaves are
// added by the balanced tree over their index, in FP64 (host replica:
// icp_sum_records).  32 lanes read the 128 bytes of one record.
// Step: wavefront 0 holds row i of the 6x6 system in lane i; each operation is
// icp_step's and se3_exp's own, in the same order, but a column's entries (and
// an element each of the 4x4 products) are computed side by side, and the
// pose block is read once into LDS at the start and written once.  Bound by the
// chain of dependent FP64 operations and loads: about 6 us.  One thread doing
// all of it, with a memory round trip for each pose entry it changed, took 11
// to 13 us.
// Tinc <- exp(xi) Tinc.  On the session's last iteration of the frame apply
// the reference's guard (gnSolver.cu:426-428) and set T = Tprev * Tinc.
__device__ void icp_finish(const DmView &v, int level, int it, int nwg, IcpStepLds &S) {
  const int k = threadIdx.x & 31, j = threadIdx.x >> 5;
  if (threadIdx.x < PD_COUNT) S.pd[threadIdx.x] = v.posed[threadIdx.x];
  // the session's parameters, on their way with the records
  const float lambda = v.lambda, min_inc = v.min_inc, max_inc = v.max_inc;
  bool last = it == v.iters[level], none = true;  // none: no finer level takes iterations
  for (int l = 0; l < level; ++l) none = none && v.iters[l] == 0;
  auto value = [&](int t) { return record_value(v.partials + (size_t)min(t, nwg - 1) * kIcpVals + k); };
#pragma unroll 1
  for (int h = 0; h < 2; ++h) {  // leaves 128 h .. 128 h + 127
    // every load unconditional (past the end: the last record, not added), so
    // that 16 are in flight together
    float x[2][8];
    const int t0 = 128 * h + 8 * j;
    if (128 * h < nwg) {
#pragma unroll
      for (int q = 0; q < 16; ++q) x[q >> 3][q & 7] = value(t0 + 64 * (q >> 3) + (q & 7));
    }
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      double l[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) l[q] = t0 + 64 * g + q < nwg ? 0.0 + (double)x[g][q] : 0.0;
      for (int t = t0 + 64 * g + 256; t < nwg; t += 256) {  // more than 256 records (512x512 pixels)
#pragma unroll
        for (int q = 0; q < 8; ++q) x[g][q] = value(t + q);
#pragma unroll
        for (int q = 0; q < 8; ++q) l[q] = t + q < nwg ? l[q] + (double)x[g][q] : l[q];
      }
      S.part[16 * h + 8 * g + j][k] = ((l[0] + l[1]) + (l[2] + l[3])) + ((l[4] + l[5]) + (l[6] + l[7]));
    }
  }
  __syncthreads();
  if (threadIdx.x >= 64) return;
  const int lane = threadIdx.x;
  double part[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    double l[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) l[q] = S.part[8 * g + q][k];
    part[g] = ((l[0] + l[1]) + (l[2] + l[3])) + ((l[4] + l[5]) + (l[6] + l[7]));
  }
  const double sum = (part[0] + part[1]) + (part[2] + part[3]);
  // icp_step: row `lane` of A (lanes 0..5), scaled by 1 / max(A), damped
  const double s0 = lane_f64(sum, 0);
  double mx = half_max(lane < 21 ? sum : s0);
  mx = s0 != s0 ? s0 : lane_f64(mx, 0);
  double xi[6] = {0, 0, 0, 0, 0, 0};
  if (mx > 0.0) {
    const double sc = 1.0 / mx;
    const double alpha = (double)lambda * (mx * sc) / (double)it;
    const int row = lane < 6 ? lane : 5;
    double A[6], L[6], D[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      const int r0 = min(row, c), c0 = max(row, c);
      A[c] = __shfl(sum, 6 * r0 - (r0 * (r0 - 1)) / 2 + c0 - r0, 64) * sc;
      if (c == row) A[c] += alpha;
    }
    double y = -__shfl(sum, 21 + row, 64) * sc;
    bool ok = true;
#pragma unroll
    for (int c = 0; c < 6; ++c) {  // column c of L, one row per lane
      double d = lane_f64(A[c], c), a = A[c];
#pragma unroll
      for (int q = 0; q < c; ++q) {
        const double lc = lane_f64(L[q], c);
        d -= lc * lc * D[q];
        a -= L[q] * lc * D[q];
      }
      D[c] = d;
      ok = ok && d > 0.0;
      L[c] = a / d;
    }
#pragma unroll
    for (int q = 0; q < 5; ++q) {  // forward substitution
      const double yq = lane_f64(y, q);
      if (row > q) y -= L[q] * yq;
    }
    double dr = D[0];
#pragma unroll
    for (int q = 1; q < 6; ++q) dr = row == q ? D[q] : dr;
    y /= dr;
#pragma unroll
    for (int i = 5; i >= 0; --i) {  // back substitution
      double a = lane_f64(y, i);
#pragma unroll
      for (int q = i + 1; q < 6; ++q) a -= lane_f64(L[i], q) * xi[q];
      xi[i] = a;
    }
    if (!ok)
#pragma unroll
      for (int q = 0; q < 6; ++q) xi[q] = 0.0;
  }
  double E[16];
  se3_exp(xi, E);
  const int r4 = (lane >> 2) & 3, c4 = lane & 3, e = lane & 15;
#pragma unroll
  for (int q = 0; q < 16; ++q)
    if (e == q) S.m[q] = E[q];
  wave_lds();
  const double *Ti = S.pd + PD_TINC;
  double tinc = S.m[4 * r4] * Ti[c4] + S.m[4 * r4 + 1] * Ti[4 + c4] + S.m[4 * r4 + 2] * Ti[8 + c4] +
                S.m[4 * r4 + 3] * Ti[12 + c4];
  // gnSolver.cu:413-415: the level ends once the summed twist changed by at
  // most min_increment since the last step that did not end a level
  double acc[6], prev[6];
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    acc[q] = S.pd[PD_ACC + q] + xi[q];
    prev[q] = S.pd[PD_PREVACC + q];
  }
  const bool stop = level_converged(acc, prev, (double)min_inc);
#pragma unroll
  for (int q = 0; q < 6; ++q)
    if (lane == q) {
      v.posed[PD_ACC + q] = acc[q];
      v.posed[PD_PREVACC + q] = prev[q];
    }
  if (stop && lane == 0) v.ctr[C_ICP_STOP] = level + 1;
  last = (last || stop) && none;
  if (last) {
    const double ssum = acc[0] + acc[1] + acc[2] + acc[3] + acc[4] + acc[5];
    if (ssum != ssum || isinf(ssum) || ssum >= (double)max_inc) {
      tinc = r4 == c4 ? 1.0 : 0.0;
      if (lane == 0) atomicAdd(&v.ctr[C_ICP_FAIL], 1);
    }
    if (lane < 16) S.t[e] = tinc;
    wave_lds();
    const double *Tp = S.pd + PD_TPREV;
    const double T = Tp[4 * r4] * S.t[c4] + Tp[4 * r4 + 1] * S.t[4 + c4] + Tp[4 * r4 + 2] * S.t[8 + c4] +
                     Tp[4 * r4 + 3] * S.t[12 + c4];
    const double Tf = (double)(float)T;  // the inverse is the float pose's
    if (lane < 16) S.m[e] = Tf;  // its last readers are before the wave_lds above
    wave_lds();
    const double inv = r4 == 3 ? (c4 == 3 ? 1.0 : 0.0)
                       : c4 < 3 ? S.m[4 * c4 + r4]
                                : -(S.m[r4] * S.m[3] + S.m[4 + r4] * S.m[7] + S.m[8 + r4] * S.m[11]);
    if (lane < 16) {
      v.posed[PD_T + e] = T;
      v.posef[PF_T + e] = (float)T;
      v.posef[PF_TINV + e] = (float)inv;
    }
  }
  if (lane < 16) {
    v.posed[PD_TINC + e] = tinc;
    v.posef[PF_TINC + e] = (float)tinc;
  }
}

// Value k of the workgroup's record into v.partials, then, with solve, the
// step by the workgroup that is the session's last to do so (threads < kVals
// call with their value, the others with any; all threads call).
// Records and tickets pass between XCDs, whose L2s are not coherent within a
// launch.  A device-scope release would write back the whole L2 (about 0.5 us
// each, serialised per XCD: 4800 workgroups lost 0.28 ms to it); instead the
// record is stored write-through (agent-scope atomic stores), wavefront 0 waits
// for its stores to complete there, and only then takes its ticket; the last
// one reads the records past its caches.  Tickets of one counter are served
// about 80 ns apart (300 workgroups: 24 us), so the workgroups of a group of 16
// count among themselves, in an unused value of the group's first record, and
// each group's last one counts for the session.
// The step in the reduction's launch saves a launch per iteration, most of
// them no-ops because the level has converged.  A full iteration of one session
// took, as reduction + step with the pixels' loads behind their tests, 13.4 + 9.0 us
// at 640x480 with the photometric term (11.2 + 8.7 without) and 10.7 + 9.0 us at
// 80x60; now 17.4 (15.3) and 14.1 us in one launch.
constexpr int kIcpGroup = 16;
__device__ __forceinline__ void icp_record(const DmView &v, float val, int level, int it, int nwg, int solve,
                                           IcpStepLds &S) {
  if (threadIdx.x < kVals)
    __hip_atomic_store(v.partials + (size_t)blockIdx.x * kIcpVals + threadIdx.x, val, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  if (!solve) return;
  __shared__ int last;
  if (threadIdx.x < 64) {  // the wavefront that stored the record
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (threadIdx.x == 0) {
      const int g = blockIdx.x / kIcpGroup, ng = (nwg + kIcpGroup - 1) / kIcpGroup;
      int *gt = (int *)(v.partials + (size_t)g * kIcpGroup * kIcpVals + 31);
      int l = 0;
      if (__hip_atomic_fetch_add(gt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
          min(kIcpGroup, nwg - g * kIcpGroup) - 1) {
        __hip_atomic_store(gt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        l = ng == 1 ||
            __hip_atomic_fetch_add(&v.ctr[C_TICKET], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == ng - 1;
      }
      last = l;
    }
  }
  __syncthreads();
  if (!last) return;
  if (threadIdx.x == 0) v.ctr[C_TICKET] = 0;
  icp_finish(v, level, it, nwg, S);
}

// One linearisation: every thread accumulates 4 pixels (strided by 256 for
// coalescing) in FP32; a wavefront tree (wave_sum: DPP row permutes, then
// two shuffles) and an LDS stage reduce them to one record per workgroup.
__global__ __launch_bounds__(256) void k_icp_reduce(const DmView *__restrict__ views, const int *__restrict__ active,
                                                     int level, int it, int solve) {
  const int slot_ = active[blockIdx.y];
  if (slot_ < 0) return;
  const DmView &v = views[slot_];
  if (v.ctr[C_HAS_MODEL] == 0 || it > v.iters[level] || v.ctr[C_ICP_STOP] == level + 1) return;
  const Intr s = level_intr(v, level);
  const int P = s.rows * s.cols;
  const int nwg = icp_wg_count(P);
  if ((int)blockIdx.x >= nwg) return;
  float vals[kVals];
#pragma unroll
  for (int k = 0; k < kVals; ++k) vals[k] = 0.f;
  IcpPose T;
  IcpPixel px[kIcpPer];
  icp_pixels(v, level, s, P, T, px);
#pragma unroll
  for (int q = 0; q < kIcpPer; ++q) icp_terms(v, s, T, px[q], vals);
  // wavefront tree (wave_sum) then LDS across the four waves
#pragma unroll
  for (int k = 0; k < kVals; ++k) vals[k] = wave_sum(vals[k]);
  __shared__ float red[4][kVals];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < kVals; ++k) red[wave][k] = vals[k];
  }
  __syncthreads();
  float val = 0.f;
  if (threadIdx.x < kVals) {
    const int k = threadIdx.x;
    val = (red[0][k] + red[1][k]) + (red[2][k] + red[3][k]);
  }
  __shared__ IcpStepLds step;
  icp_record(v, val, level, it, nwg, solve, step);
}

// The same linearisation on the matrix cores: each pixel's 16-float feature
// row (icp_features) is staged through LDS and v_mfma_f32_16x16x4f32
// accumulates F^T F over 4 rows per instruction (lane l supplies feature l %
// 16 of row l / 16 as both operands; the 16x16 result holds column l % 16,
// rows 4 (l / 16) .. + 3 in lane l).  The four waves' tiles are added in a
// fixed order and the record takes J^T J = G + P (the geometric and
// photometric 6x6 blocks), J^T r, the counts and r^2 from the tile.  Same
// grid and record layout as k_icp_reduce; the sums differ from it by
// rounding only (w_photo enters as sqrt(w_photo)^2).
typedef float icp_f4 __attribute__((ext_vector_type(4)));
constexpr int kFeatPitch = 17;  // LDS row pitch (floats): rows of a wave fall on distinct banks
__global__ __launch_bounds__(256) void k_icp_reduce_mfma(const DmView *__restrict__ views,
                                                          const int *__restrict__ active, int level, int it,
                                                          int solve) {
  const int slot_ = active[blockIdx.y];
  if (slot_ < 0) return;
  const DmView &v = views[slot_];
  if (v.ctr[C_HAS_MODEL] == 0 || it > v.iters[level] || v.ctr[C_ICP_STOP] == level + 1) return;
  const Intr s = level_intr(v, level);
  const int P = s.rows * s.cols;
  const int nwg = icp_wg_count(P);
  if ((int)blockIdx.x >= nwg) return;
  __shared__ float feat[4][64 * kFeatPitch];
  __shared__ float tile[4][256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float *F = feat[wave];
  const float swp = v.w_photo > 0.f ? sqrtf(v.w_photo) : 0.f;
  icp_f4 acc = {0.f, 0.f, 0.f, 0.f};
  IcpPose T;
  IcpPixel px[kIcpPer];
  icp_pixels(v, level, s, P, T, px);
#pragma unroll
  for (int q = 0; q < kIcpPer; ++q) {
    float f[16];
    icp_features(v, s, T, px[q], swp, f);
#pragma unroll
    for (int k = 0; k < 16; ++k) F[lane * kFeatPitch + k] = f[k];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 16; ++m) {
      const float a = F[(4 * m + (lane >> 4)) * kFeatPitch + (lane & 15)];
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a, a, acc, 0, 0, 0);
    }
    __syncthreads();  // the rows are rewritten by the next group of pixels
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) tile[wave][(4 * (lane >> 4) + e) * 16 + (lane & 15)] = acc[e];
  __syncthreads();
  float val = 0.f;
  if (threadIdx.x < kVals) {
    const int k = threadIdx.x;
    auto T = [&](int r, int c) {
      const int o = r * 16 + c;
      return (tile[0][o] + tile[1][o]) + (tile[2][o] + tile[3][o]);
    };
    if (k < 21) {
      int a = 0, kk = k;
      while (kk >= 6 - a) { kk -= 6 - a; ++a; }
      const int b = a + kk;
      val = T(a, b) + T(8 + a, 8 + b);
    } else if (k < 27) {
      val = T(k - 21, 6) + T(8 + (k - 21), 14);
    } else if (k == 27) {
      val = T(7, 7);
    } else if (k == 28) {
      val = T(6, 6);
    } else {
      val = T(15, 15);
    }
  }
  __shared__ IcpStepLds step;
  icp_record(v, val, level, it, nwg, solve, step);
}

// Start of a frame: Tprev <- T when a model exists, otherwise T <- Tinit;
// Tinc <- I, summed twist <- 0.
__global__ void k_pose_begin(const DmView *__restrict__ views, const int *__restrict__ active) {
  const int slot_ = active[blockIdx.x];
  if (slot_ < 0) return;
  const DmView &v = views[slot_];
  if (threadIdx.x != 0) return;
  double *P = v.posed;
  if (v.ctr[C_HAS_MODEL]) {
    for (int k = 0; k < 16; ++k) P[PD_TPREV + k] = P[PD_T + k];
  } else {
    for (int k = 0; k < 16; ++k) P[PD_T + k] = P[PD_TINIT + k];
  }
  for (int k = 0; k < 16; ++k) {
    v.posef[PF_T + k] = (float)P[PD_T + k];
    v.posef[PF_TPREV + k] = (float)P[PD_TPREV + k];
    P[PD_TINC + k] = (k % 5 == 0) ? 1.0 : 0.0;
    v.posef[PF_TINC + k] = (k % 5 == 0) ? 1.f : 0.f;
  }
  rigid_inverse_ff(v.posef + PF_T, v.posef + PF_TINV);
  for (int k = 0; k < 6; ++k) P[PD_ACC + k] = 0.0;
  for (int k = 0; k < 6; ++k) P[PD_PREVACC + k] = 0.0;
  v.ctr[C_ICP_STOP] = 0;
  v.ctr[C_NVIS] = 0;
  v.ctr[C_NVISIT] = 0;
}

struct PoseArg { float T[16], Ti[16]; };
__global__ __launch_bounds__(256) void k_set_view(DmView *__restrict__ dst, DmView h, PoseArg p, int set_pose) {
  const int t = threadIdx.x;
  static_assert(sizeof(DmView) % 8 == 0 && sizeof(DmView) / 8 <= 256, "one word per thread");
  if (t < (int)(sizeof(DmView) / 8)) ((uint64_t *)dst)[t] = ((const uint64_t *)&h)[t];
  if (set_pose && t < 16) {
    h.posef[PF_T + t] = p.T[t];
    h.posef[PF_TINV + t] = p.Ti[t];
    h.posed[PD_T + t] = (double)p.T[t];
  }
}
void launch_set_view(DmView *d_view, const DmView &h, const float *pose, hipStream_t st) {
  PoseArg p{};
  if (pose) {
    for (int k = 0; k < 16; ++k) p.T[k] = pose[k];
    rigid_inverse_ff(p.T, p.Ti);
  }
  hipLaunchKernelGGL(k_set_view, dim3(1), dim3(256), 0, st, d_view, h, p, pose ? 1 : 0);
}

__global__ __launch_bounds__(128) void k_track_reset(double *__restrict__ posed, float *__restrict__ posef,
                                                     int32_t *__restrict__ ctr) {
  const int t = threadIdx.x;
  if (t < PD_COUNT) {
    const bool mat = t < PD_ACC || (t >= PD_TINIT && t < PD_PERSIST);
    posed[t] = mat && (t & 15) % 5 == 0 ? 1.0 : 0.0;
  }
  if (t < PF_COUNT) posef[t] = (t & 15) % 5 == 0 ? 1.f : 0.f;
  if (t == 0) {
    ctr[C_HAS_MODEL] = 1;
    ctr[C_ICP_STOP] = 0;
  }
}
void launch_track_reset(const DmView &h, hipStream_t st) {
  static_assert(PD_T % 16 == 0 && PD_TPREV % 16 == 0 && PD_TINC % 16 == 0 && PD_TINIT % 16 == 0 && PD_COUNT <= 128,
                "matrices at multiples of 16");
  hipLaunchKernelGGL(k_track_reset, dim3(1), dim3(128), 0, st, h.posed, h.posef, h.ctr);
}

__global__ __launch_bounds__(256) void k_pack_maps(const float4 *__restrict__ vert, const float4 *__restrict__ norm,
                                                   int n, float *__restrict__ v3, float *__restrict__ n3,
                                                   float *__restrict__ inten) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  if (v3 || inten) {
    const float4 a = vert[i];
    if (v3) { v3[3 * i] = a.x; v3[3 * i + 1] = a.y; v3[3 * i + 2] = a.z; }
    if (inten) inten[i] = a.w;
  }
  if (n3) {
    const float4 a = norm[i];
    n3[3 * i] = a.x; n3[3 * i + 1] = a.y; n3[3 * i + 2] = a.z;
  }
}
void launch_pack_maps(const float4 *vert, const float4 *norm, int n, float *v3, float *n3, float *inten,
                      hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_pack_maps, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, vert, norm, n, v3, n3, inten);
}

void launch_source_maps(const Launch &L) {
  if (L.nact <= 0) return;
  const int tot = L.max_pixels + L.max_pixels / 4 + L.max_pixels / 16 + 2;
  hipLaunchKernelGGL(k_source_maps, dim3((unsigned)((tot + 255) / 256), (unsigned)L.nact), dim3(256), 0, L.stream,
                     L.views, L.active);
}

void launch_icp_reduce(const Launch &L, int level, int it, bool solve) {
  if (L.nact <= 0) return;
  const int P = L.max_pixels >> (2 * level);
  hipLaunchKernelGGL(L.icp_mfma ? k_icp_reduce_mfma : k_icp_reduce, dim3((unsigned)icp_wg_count(P), (unsigned)L.nact),
                     dim3(256), 0, L.stream, L.views, L.active, level, it, solve ? 1 : 0);
}

void icp_sum_records(const float *part, int nwg, double *sums) {
  for (int k = 0; k < kVals; ++k) {
    double lane[256];
    for (int t = 0; t < 256; ++t) {
      double a = 0.0;
      for (int w = t; w < nwg; w += 256) a += (double)part[(size_t)w * kIcpVals + k];
      lane[t] = a;
    }
    // wave_sum's steps: lane i adds lane src(i) for src = i ^ 1, i ^ 2, the
    // half-row mirror, the row mirror, i ^ 16, i ^ 32
    auto src = [](int step, int i) {
      switch (step) {
        case 0: return i ^ 1;
        case 1: return i ^ 2;
        case 2: return (i & ~7) | (7 - (i & 7));
        case 3: return (i & ~15) | (15 - (i & 15));
        case 4: return i ^ 16;
        default: return i ^ 32;
      }
    };
    double wv[4];
    for (int q = 0; q < 4; ++q) {
      double x[64];
      for (int i = 0; i < 64; ++i) x[i] = lane[64 * q + i];
      for (int step = 0; step < 6; ++step) {
        double y[64];
        for (int i = 0; i < 64; ++i) y[i] = x[i] + x[src(step, i)];
        for (int i = 0; i < 64; ++i) x[i] = y[i];
      }
      wv[q] = x[0];
    }
    sums[k] = (wv[0] + wv[1]) + (wv[2] + wv[3]);
  }
}

void launch_pose_begin(const Launch &L) {
  if (L.nact <= 0) return;
  hipLaunchKernelGGL(k_pose_begin, dim3((unsigned)L.nact), dim3(64), 0, L.stream, L.views, L.active);
}

// Copy the frame pose of every session of a batch into a log (dest[y] is the
// log row of list entry y).
__global__ void k_pose_log(const DmView *__restrict__ views, const int *__restrict__ active,
                           const int *__restrict__ dest, double *__restrict__ log) {
  const int slot_ = active[blockIdx.x];
  if (slot_ < 0) return;
  const DmView &v = views[slot_];
  if (threadIdx.x < 16) log[(size_t)dest[blockIdx.x] * 16 + threadIdx.x] = v.posed[PD_T + threadIdx.x];
}

void launch_pose_log(const Launch &L, const int *dest, double *log) {
  if (L.nact <= 0) return;
  hipLaunchKernelGGL(k_pose_log, dim3((unsigned)L.nact), dim3(64), 0, L.stream, L.views, L.active, dest, log);
}


}  // namespace dm
