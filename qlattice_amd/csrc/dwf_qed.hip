// The QED domain-wall operator on full (not even-odd) 5D fields [site][s][4]
// (multiply_m_dwf_qed, qed.cpp:263-411) and the vector updates of its CG.
#include "dwf_internal.h"
#include "dwf_rules.h"

namespace qdwf {

__device__ __forceinline__ double2 zmul(double2 a, double2 b)
{
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 zconj_if(bool c, double2 a) { return make_double2(a.x, c ? -a.y : a.y); }
__device__ __forceinline__ double2 zaxpy(double a, double2 x, double2 y)
{
  return make_double2(y.x + a * x.x, y.y + a * x.y);
}

// inv[i] = 1 / gf[i]
__global__ void __launch_bounds__(kBlasBlock) k_qed_inverse(const double2* __restrict__ gf, double2* __restrict__ inv,
                                                            int64_t n)
{
  for (int64_t i = (int64_t)blockIdx.x * kBlasBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlasBlock) {
    const double2 g = gf[i];
    const double d = g.x * g.x + g.y * g.y;
    inv[i] = make_double2(g.x / d, -g.y / d);
  }
}
void launch_qed_inverse(const double2* gf, double2* inv, int64_t n, hipStream_t st)
{
  hipLaunchKernelGGL(k_qed_inverse, dim3(blas_grid(n)), dim3(kBlasBlock), 0, st, gf, inv, n);
}

// the value of the quad's lane r ^ X, X = 2 or 3
template <int X>
__device__ __forceinline__ double quad_xor(double d)
{
  constexpr int kPerm = X == 3 ? 0x1B : 0x4E;  // quad_perm [3,2,1,0] or [2,3,0,1]
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(d), kPerm, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(d), kPerm, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}
template <int X>
__device__ __forceinline__ double2 quad_xor(double2 v)
{
  return make_double2(quad_xor<X>(v.x), quad_xor<X>(v.y));
}

// One thread per element (site, s, spin r): every load of a wave is one
// contiguous run of the field, and the other spin of a gamma comes from the
// quad's lanes.  The CPS gammas (matrix.h:426-452) have one non-zero per row:
// column r ^ 3 for x and y, r ^ 2 for z and t.  The links' inverses (the
// backward link is 1 / gf1(x - mu)) are formed once per call.
// Latency bound on the lattices it runs on: 8^3x16 Ls8 8.3 us, and 30.5 us with
// one thread per (site, s), its 64-byte strided loads and its 4 to 13 FP64
// divisions.
template <bool DAG, bool DOT>
__global__ void __launch_bounds__(kBlasBlock) k_qed_m(QedArgs a)
{
  if (a.cg && a.cg->done) return;
  const int64_t blk = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
  if (blk * kBlasBlock >= a.nelem) return;  // (of a grid spread over y)
  const int64_t i = blk * kBlasBlock + threadIdx.x;
  double dot = 0.0;
  if (i < a.nelem) {
    const int ls = a.ls, r = (int)(i & 3);
    const int64_t j = i >> 2;
    int64_t site;
    int x[4];
    if (a.nelem < (int64_t)1 << 33) {  // (uniform) j below 2^31
      unsigned q = fdiv((unsigned)j, a.dls);
      site = q;
#pragma unroll
      for (int mu = 0; mu < 3; ++mu) {
        const unsigned t = fdiv(q, a.dn[mu]);
        x[mu] = (int)(q - t * (unsigned)a.n[mu]);
        q = t;
      }
      x[3] = (int)q;
    } else {
      int64_t q = site = j / ls;
#pragma unroll
      for (int mu = 0; mu < 3; ++mu) {
        x[mu] = (int)(q % a.n[mu]);
        q /= a.n[mu];
      }
      x[3] = (int)q;
    }
    const int s = (int)(j - site * ls);
    // Wick phase factors of the time slice: (tw + twm)/2, (1/tw + 1/twm)/2,
    // 1/tw, 1/twm with twm = tw(t - 1)
    double2 avg = make_double2(1.0, 0.0), iavg = avg, itw = avg, itwm = avg;
    if (a.wick) {
      avg = zconj_if(DAG, a.wick[4 * x[3]]);
      iavg = zconj_if(DAG, a.wick[4 * x[3] + 1]);
      itw = zconj_if(DAG, a.wick[4 * x[3] + 2]);
      itwm = zconj_if(DAG, a.wick[4 * x[3] + 3]);
    }
    const double df = DAG ? -1.0 : 1.0, g5 = r < 2 ? 1.0 : -1.0;
    auto at = [&](int64_t st, int ss) { return a.in[((st * ls + ss) << 2) + r]; };
    double2 v = zmul(make_double2((4.0 - a.m5) * avg.x + iavg.x, (4.0 - a.m5) * avg.y + iavg.y), at(site, s));
    // fifth dimension (qed.cpp:342-371)
    double2 f = make_double2(0.0, 0.0);
    if (s < ls - 1) f = zaxpy(-0.5 + df * 0.5 * g5, at(site, s + 1), f);
    if (s > 0) f = zaxpy(-0.5 - df * 0.5 * g5, at(site, s - 1), f);
    if (s == ls - 1) f = zaxpy(0.5 * a.mass * (1.0 - df * g5), at(site, 0), f);
    if (s == 0) f = zaxpy(0.5 * a.mass * (1.0 + df * g5), at(site, ls - 1), f);
    // hopping (qed.cpp:373-408): -1/2 U(x) (tf2 - df tf1 G) in(x+mu) and
    // -1/2 U^-1(x-mu) (tfm2 + df tfm1 G) in(x-mu); tf1 = tf2 = avg for mu < 3
    const double sgn[3] = {r < 2 ? 1.0 : -1.0, (r == 1 || r == 2) ? 1.0 : -1.0, (r == 0 || r == 3) ? 1.0 : -1.0};
    int64_t stride = 1;
#pragma unroll
    for (int mu = 0; mu < 4; ++mu) {
      const int L = a.n[mu];
      const int64_t sp = site + (x[mu] + 1 == L ? -(int64_t)(L - 1) : 1) * stride;
      const int64_t sm = site + (x[mu] == 0 ? (int64_t)(L - 1) : -1) * stride;
      stride *= L;
      const double2 up = DAG ? zconj_if(true, a.gfi[site * 4 + mu]) : a.gf[site * 4 + mu];
      const double2 um = DAG ? zconj_if(true, a.gf[sm * 4 + mu]) : a.gfi[sm * 4 + mu];
      const double2 wp = at(sp, s), wm = at(sm, s);
      double2 gp, gm;
      if (mu < 2) {
        gp = quad_xor<3>(wp);
        gm = quad_xor<3>(wm);
      } else {
        gp = quad_xor<2>(wp);
        gm = quad_xor<2>(wm);
      }
      if (mu == 0 || mu == 2) {
        gp = make_double2(-sgn[mu] * gp.y, sgn[mu] * gp.x);
        gm = make_double2(-sgn[mu] * gm.y, sgn[mu] * gm.x);
      } else if (mu == 1) {
        gp = make_double2(sgn[1] * gp.x, sgn[1] * gp.y);
        gm = make_double2(sgn[1] * gm.x, sgn[1] * gm.y);
      }
      if (mu < 3) {
        f = zaxpy(-0.5, zmul(up, zaxpy(-df, gp, wp)), f);
        f = zaxpy(-0.5, zmul(um, zaxpy(df, gm, wm)), f);
      } else {
        v = zaxpy(-0.5, zmul(up, zaxpy(-df, gp, zmul(itw, wp))), v);
        v = zaxpy(-0.5, zmul(um, zaxpy(df, gm, zmul(itwm, wm))), v);
      }
    }
    const double2 af = zmul(avg, f);
    v = make_double2(v.x + af.x, v.y + af.y);
    a.out[i] = v;
    if (DOT) {
      const double2 p = a.dotp[i];
      dot = p.x * v.x + p.y * v.y;
    }
  }
  if (DOT) {
    dot = block_sum<kBlasBlock / 64>(dot);
    if (threadIdx.x == 0) a.part[blk] = dot;
  }
}

int64_t qed_m_blocks(const QedArgs& a) { return (a.nelem + kBlasBlock - 1) / kBlasBlock; }

void launch_qed_m(const QedArgs& a, hipStream_t st)
{
  const Grid2 g = split_blocks(qed_m_blocks(a), kBlasBlock);
  const dim3 grid(g.x, g.y), blk(kBlasBlock);
  if (a.dagger) {
    if (a.dotp) hipLaunchKernelGGL((k_qed_m<true, true>), grid, blk, 0, st, a);
    else hipLaunchKernelGGL((k_qed_m<true, false>), grid, blk, 0, st, a);
  } else {
    if (a.dotp) hipLaunchKernelGGL((k_qed_m<false, true>), grid, blk, 0, st, a);
    else hipLaunchKernelGGL((k_qed_m<false, false>), grid, blk, 0, st, a);
  }
}

// The vector updates of one CG iteration, scalars on the device as in
// k_cg_residual_d / k_cg_step_d: x += alpha p, r -= alpha ap; p = r + beta p.
__global__ void __launch_bounds__(256) k_qed_update(QedIterArgs a)
{
  CgState64* st = a.st + a.slot;
  if (st->done) return;
  const double alpha = st->rr / sum_parts(a.pap, a.npap);
  double v = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < a.n; i += (int64_t)gridDim.x * 256) {
    a.x[i] = zaxpy(alpha, a.p[i], a.x[i]);
    const double2 r = zaxpy(-alpha, a.ap[i], a.r[i]);
    a.r[i] = r;
    v += r.x * r.x + r.y * r.y;
  }
  __syncthreads();  // the sum's LDS is reused
  v = block_sum<4>(v);
  if (threadIdx.x == 0) a.rnorm[blockIdx.x] = v;
}

__global__ void __launch_bounds__(256) k_qed_direction(QedIterArgs a, int nrnorm)
{
  const CgState64 st = a.st[a.slot];
  const bool first = blockIdx.x == 0 && threadIdx.x == 0;
  if (st.done) {  // the state is carried on for the iterations queued behind
    if (first) a.st[1 - a.slot] = st;
    return;
  }
  const double rr = sum_parts(a.rnorm, nrnorm);
  const CgState64 next{rr, st.target, 0.0, st.iter + 1, !isfinite(rr) ? 2 : rr <= st.target ? 1 : 0};
  if (first) {
    a.st[1 - a.slot] = next;
    *a.host = next;
  }
  if (next.done) return;
  const double beta = rr / st.rr;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < a.n; i += (int64_t)gridDim.x * 256)
    a.p[i] = zaxpy(beta, a.p[i], a.r[i]);
}

void launch_qed_iter(const QedIterArgs& a, hipStream_t st)
{
  const int g = cg_residual_grid(a.n);
  hipLaunchKernelGGL(k_qed_update, dim3(g), dim3(256), 0, st, a);
  hipLaunchKernelGGL(k_qed_direction, dim3(g), dim3(256), 0, st, a, g);
}

// 4D [site][4] -> 5D [site][s][4]: spins 0, 1 at s = 0 and 2, 3 at s = ls - 1
// (fermion_field_5d_from_4d_qed), and back from the opposite walls.
__global__ void __launch_bounds__(kBlasBlock) k_qed_embed(const double2* __restrict__ in, double2* __restrict__ out,
                                                          int ls, int64_t n)
{
  for (int64_t i = (int64_t)blockIdx.x * kBlasBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlasBlock) {
    const int64_t j = i >> 2, site = j / ls;
    const int r = (int)(i & 3), s = (int)(j - site * ls);
    out[i] = s == (r < 2 ? 0 : ls - 1) ? in[site * 4 + r] : make_double2(0.0, 0.0);
  }
}
__global__ void __launch_bounds__(kBlasBlock) k_qed_project(const double2* __restrict__ in, double2* __restrict__ out,
                                                            int ls, int64_t n4)
{
  for (int64_t i = (int64_t)blockIdx.x * kBlasBlock + threadIdx.x; i < n4; i += (int64_t)gridDim.x * kBlasBlock) {
    const int r = (int)(i & 3);
    out[i] = in[((i >> 2) * ls + (r < 2 ? ls - 1 : 0)) * 4 + r];
  }
}
void launch_qed_embed(const double2* in4, double2* out5, int ls, int64_t vol, hipStream_t st)
{
  const int64_t n = vol * ls * 4;
  hipLaunchKernelGGL(k_qed_embed, dim3(blas_grid(n)), dim3(kBlasBlock), 0, st, in4, out5, ls, n);
}
void launch_qed_project(const double2* in5, double2* out4, int ls, int64_t vol, hipStream_t st)
{
  const int64_t n4 = vol * 4;
  hipLaunchKernelGGL(k_qed_project, dim3(blas_grid(n4)), dim3(kBlasBlock), 0, st, in5, out4, ls, n4);
}

}  // namespace qdwf
