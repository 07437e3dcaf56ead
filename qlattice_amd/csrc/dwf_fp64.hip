// FP64 kernels of the domain-wall operators: the Wilson hop, the hop fused
// with a fifth-dimension (s) matrix, the s-matrices alone and the CG step.
// The s-matrices run on the matrix cores (v_mfma_f64_16x16x4_f64).
#include "dwf_internal.h"

namespace qdwf {

typedef double mf4d __attribute__((ext_vector_type(4)));

// Inputs that a kernel reads once: non-temporal loads where a field is far
// beyond the 256 MB last-level cache (24^3x64 Ls12, 1 GB: the hop with x
// 0.96 -> 0.94 ms, the s-matrix 0.453 -> 0.431 ms), ordinary ones below,
// where the previous kernel's output is still cached (with non-temporal
// loads the hop with x took 100 instead of 90 us at 16^3x32 Ls8 and 13.3
// instead of 8.9 us at 8^3x16).
static bool stream_field(const LatGeo& g, int ls) { return (int64_t)ls * 192 * g.stride > (int64_t)512 << 20; }

// ------------------------------------------------- s-matrix products
// out(s) = sum_t M_chi[s][t] in(t), per real component a (rows s, in tiles of
// 16) x (t, in steps of 4) by (t) x (16 sites) product.  Lane l of a wave
// supplies A[s = 16 mt + l%16][t = 4 kb + l/16] (the matrix) and
// B[t = 4 kb + l/16][site = l%16], and receives D[s = 16 mt + l/16 + 4 i]
// [site = l%16], i < 4.  A double2 slot of the field (re, im of one
// component) feeds the B operands of two products, so that lane l reads and
// writes the field at (site l%16, one t or s): 16 sites are one 256-byte run
// of the blocked layout on either side, and a lane ends up with whole slots.
// Rows and columns beyond ls are zero operands.
template <int LSMAX, bool REAL>
struct SMat {
  static constexpr int MT = (LSMAX + 15) / 16, KB = (LSMAX + 3) / 4;
  double re[MT][KB], im[REAL ? 1 : MT][REAL ? 1 : KB];
  __device__ __forceinline__ void load(const cplx<double>* __restrict__ m, int ls)
  {
    const int li = threadIdx.x & 15, lq = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const int s = mt * 16 + li, t = 4 * kb + lq;
        cplx<double> v = cmk<double>(0, 0);
        if (s < ls && t < ls) v = m[s * ls + t];
        re[mt][kb] = v.re;
        if constexpr (!REAL) im[mt][kb] = v.im;
      }
  }
  // dr, di += M column step kb times b
  __device__ __forceinline__ void fma(int kb, double2 b, mf4d dr[MT], mf4d di[MT]) const
  {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      dr[mt] = __builtin_amdgcn_mfma_f64_16x16x4f64(re[mt][kb], b.x, dr[mt], 0, 0, 0);
      di[mt] = __builtin_amdgcn_mfma_f64_16x16x4f64(re[mt][kb], b.y, di[mt], 0, 0, 0);
      if constexpr (!REAL) {
        dr[mt] = __builtin_amdgcn_mfma_f64_16x16x4f64(-im[mt][kb], b.y, dr[mt], 0, 0, 0);
        di[mt] = __builtin_amdgcn_mfma_f64_16x16x4f64(im[mt][kb], b.x, di[mt], 0, 0, 0);
      }
    }
  }
};

// out = alpha Mat in (+ beta x): wave = 16 sites x kSmatComps components of
// one chirality, block = 64 sites, blockIdx.y = the component group.
// HBM bound, at the speed of a copy: 0.36 to 0.42 ms at 24^3x64 Ls12 (4.9 to
// 5.7 TB/s), 30 us at 16^3x32 Ls8 and 4.3 us at 8^3x16 Ls12.  With one thread per site
// and slot looping over s on the vector units it was 0.61 ms, 46 us and
// 14.3 us (57 us at 8^3x16 Ls24: a chain of scalar loads of the matrix).
template <int LSMAX>
constexpr int kSmatComps = LSMAX <= 16 ? 3 : 1;  // (the components' operands are all in registers)
template <int LSMAX, bool XPAY, bool REAL, bool NT>
__global__ void __launch_bounds__(256) k_smat_d(M5Args<double> a)
{
  typedef SMat<LSMAX, REAL> Mx;
  constexpr int NC = kSmatComps<LSMAX>;
  const int ls = a.ls, nkb = (ls + 3) >> 2;
  const int lane = threadIdx.x & 63, li = lane & 15, lq = lane >> 4;
  const int64_t h = (int64_t)blockIdx.x * 64 + (threadIdx.x >> 6) * 16 + li;
  const int k0 = blockIdx.y * NC, chi = k0 / 6;
  const bool act = h < a.geo.vh;
  const double2* __restrict__ in = (const double2*)a.in;
  double2* __restrict__ out = (double2*)a.out;
  double2 b[NC][Mx::KB];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int kb = 0; kb < Mx::KB; ++kb) {
      const int t = 4 * kb + lq;
      b[c][kb] = make_double2(0.0, 0.0);
      if (act && t < ls) b[c][kb] = load_in<NT>(&in[sidx<12>(ls, t, k0 + c, h)]);
    }
  Mx m;
  m.load(a.mat + chi * ls * ls, ls);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    mf4d dr[Mx::MT], di[Mx::MT];
#pragma unroll
    for (int mt = 0; mt < Mx::MT; ++mt) dr[mt] = di[mt] = (mf4d){0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int kb = 0; kb < Mx::KB; ++kb)
      if (kb < nkb) m.fma(kb, b[c][kb], dr, di);
#pragma unroll
    for (int mt = 0; mt < Mx::MT; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int s = mt * 16 + lq + 4 * i;
        if (!act || s >= ls) continue;
        const unsigned o = sidx<12>(ls, s, k0 + c, h);
        double2 r = make_double2(a.alpha * dr[mt][i], a.alpha * di[mt][i]);
        if (XPAY) {
          const double2 x = load_in<NT>(&((const double2*)a.x)[o]);
          r.x += a.beta * x.x;
          r.y += a.beta * x.y;
        }
        out[o] = r;
      }
  }
}

template <int LSMAX>
static void launch_smat_ls(const M5Args<double>& a, hipStream_t st)
{
  const dim3 grid((unsigned)((a.geo.vh + 63) / 64), 12 / kSmatComps<LSMAX>);
  const dim3 blk(256);
  const bool nt = stream_field(a.geo, a.ls);
#define QDWF_L(X, R)                                                                              \
  {                                                                                               \
    if (nt) hipLaunchKernelGGL((k_smat_d<LSMAX, X, R, true>), grid, blk, 0, st, a);               \
    else hipLaunchKernelGGL((k_smat_d<LSMAX, X, R, false>), grid, blk, 0, st, a);                 \
  }
  if (a.real_mat) {
    if (a.x) QDWF_L(true, true)
    else QDWF_L(false, true)
  } else {
    if (a.x) QDWF_L(true, false)
    else QDWF_L(false, false)
  }
#undef QDWF_L
}

void launch_smat_d(const M5Args<double>& a, hipStream_t st)
{
  if (a.ls <= 8) launch_smat_ls<8>(a, st);
  else if (a.ls <= 12) launch_smat_ls<12>(a, st);
  else if (a.ls <= 16) launch_smat_ls<16>(a, st);
  else if (a.ls <= 24) launch_smat_ls<24>(a, st);
  else launch_smat_ls<32>(a, st);
}

// ------------------------------------------------------------ CG updates
// The scalars of an iteration never leave the device: each kernel sums the
// partial sums of the one before it in its blocks' prologues (always in the
// same order), so an iteration needs no reduction kernels and no host round
// trip, and the host can queue iterations ahead (cg_fp64).
__global__ void k_cg_init_d(CgState64* st, double rr, double target)
{
  st[0] = CgState64{rr, target, 0.0, 0, 0};
  st[1] = st[0];
}
void launch_cg_init_d(CgState64* st, double rr, double target, hipStream_t s)
{
  hipLaunchKernelGGL(k_cg_init_d, dim3(1), dim3(1), 0, s, st, rr, target);
}

__global__ void __launch_bounds__(256) k_cg_residual_d(CgIterDArgs a, int64_t n)
{
  CgState64* st = a.st + a.slot;
  if (st->done) return;
  const double alpha = st->rr / sum_parts(a.pap, a.npap);
  if (blockIdx.x == 0 && threadIdx.x == 0) st->alpha = alpha;  // (read by the next kernel only)
  double v = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const double2 ap = a.ap[i];
    double2 r = a.r[i];
    r.x -= alpha * ap.x;
    r.y -= alpha * ap.y;
    a.r[i] = r;
    v += r.x * r.x + r.y * r.y;
  }
  __syncthreads();  // the sum's LDS is reused
  v = block_sum<4>(v);
  if (threadIdx.x == 0) a.rnorm[blockIdx.x] = v;
}

// Mapping of k_smat_d, one component per wave; the products' operands are
// the new p, so p and t are streamed once.
template <int LSMAX, bool REAL, bool NT>
__global__ void __launch_bounds__(256) k_cg_step_d(CgIterDArgs a, int nrnorm)
{
  typedef SMat<LSMAX, REAL> Mx;
  const CgState64 st = a.st[a.slot];
  if (st.done) {  // the state is carried on for the iterations queued behind
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) a.st[1 - a.slot] = st;
    return;
  }
  const int ls = a.ls, nkb = (ls + 3) >> 2;
  const int lane = threadIdx.x & 63, li = lane & 15, lq = lane >> 4;
  const int64_t h = (int64_t)blockIdx.x * 64 + (threadIdx.x >> 6) * 16 + li;
  const int k = blockIdx.y, chi = k / 6;
  const bool act = h < a.geo.vh;
  const double rr = sum_parts(a.rnorm, nrnorm);
  const int done = !isfinite(rr) ? 2 : rr <= st.target ? 1 : 0;
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
    const CgState64 next{rr, st.target, 0.0, st.iter + 1, done};
    a.st[1 - a.slot] = next;
    *a.host = next;
  }
  const double alpha = st.alpha, beta = rr / st.rr;
  double2 b[Mx::KB];
#pragma unroll
  for (int kb = 0; kb < Mx::KB; ++kb) {
    const int t = 4 * kb + lq;
    b[kb] = make_double2(0.0, 0.0);
    if (act && t < ls) {
      const unsigned o = sidx<12>(ls, t, k, h);
      const double2 p = load_in<NT>(&a.p[o]);
      double2 x = load_in<NT>(&a.x[o]);
      x.x += alpha * p.x;
      x.y += alpha * p.y;
      a.x[o] = x;
      if (!done) {
        const double2 r = load_in<NT>(&a.r[o]);
        b[kb] = make_double2(beta * p.x + r.x, beta * p.y + r.y);
        a.p[o] = b[kb];
      }
    }
  }
  if (done) return;
  Mx m;
  m.load(a.mat + chi * ls * ls, ls);
  mf4d dr[Mx::MT], di[Mx::MT];
#pragma unroll
  for (int mt = 0; mt < Mx::MT; ++mt) dr[mt] = di[mt] = (mf4d){0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int kb = 0; kb < Mx::KB; ++kb)
    if (kb < nkb) m.fma(kb, b[kb], dr, di);
#pragma unroll
  for (int mt = 0; mt < Mx::MT; ++mt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int s = mt * 16 + lq + 4 * i;
      if (act && s < ls) a.t[sidx<12>(ls, s, k, h)] = make_double2(dr[mt][i], di[mt][i]);
    }
}

template <int LSMAX>
static void launch_cg_step_d_ls(const CgIterDArgs& a, int nrnorm, hipStream_t st)
{
  const dim3 grid((unsigned)((a.geo.vh + 63) / 64), 12);
  const bool nt = stream_field(a.geo, a.ls);
  if (a.real_mat) {
    if (nt) hipLaunchKernelGGL((k_cg_step_d<LSMAX, true, true>), grid, dim3(256), 0, st, a, nrnorm);
    else hipLaunchKernelGGL((k_cg_step_d<LSMAX, true, false>), grid, dim3(256), 0, st, a, nrnorm);
  } else {
    if (nt) hipLaunchKernelGGL((k_cg_step_d<LSMAX, false, true>), grid, dim3(256), 0, st, a, nrnorm);
    else hipLaunchKernelGGL((k_cg_step_d<LSMAX, false, false>), grid, dim3(256), 0, st, a, nrnorm);
  }
}

void launch_cg_iter_d(const CgIterDArgs& a, hipStream_t st)
{
  const int64_t n = (int64_t)a.ls * 12 * a.geo.stride;
  const int g = cg_residual_grid(n);
  hipLaunchKernelGGL(k_cg_residual_d, dim3(g), dim3(256), 0, st, a, n);
  if (a.ls <= 8) launch_cg_step_d_ls<8>(a, g, st);
  else if (a.ls <= 12) launch_cg_step_d_ls<12>(a, g, st);
  else if (a.ls <= 16) launch_cg_step_d_ls<16>(a, g, st);
  else if (a.ls <= 24) launch_cg_step_d_ls<24>(a, g, st);
  else launch_cg_step_d_ls<32>(a, g, st);
}

// r = scale (b - ax) in the solver's storage and the sums of |b - ax|^2, the
// reliable update's residual in one pass: streams b and ax and writes r
// (16^3x32 Ls12: 68 us against 200 for copy, update, norm and conversion).
template <class SR, bool NT>
__global__ void __launch_bounds__(256) k_residual_d(const double2* __restrict__ b, const double2* __restrict__ ax,
                                                    typename SpinorIO<SR>::slot_t* __restrict__ r, int ls, int64_t n5,
                                                    double scale, double* __restrict__ part)
{
  double t = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n5; i += (int64_t)gridDim.x * 256) {
    const int64_t hs = i >> 6, lane = i & 63;  // hs = (h / 64) ls + s
    const int64_t hb = (unsigned)hs / (unsigned)ls;
    const int64_t o = hs * 768 + lane;
    cplx<float> v[12];
#pragma unroll
    for (int k = 0; k < 12; ++k) {
      const double2 x = load_in<NT>(&b[o + k * 64]), y = load_in<NT>(&ax[o + k * 64]);
      const double re = x.x - y.x, im = x.y - y.y;
      t += re * re + im * im;
      v[k] = cmk<float>((float)(scale * re), (float)(scale * im));
    }
    if (r) SpinorIO<SR>::store_stream(r, ls, (int)(hs - hb * ls), (hb << 6) + lane, v);
  }
  t = block_sum<4>(t);
  if (threadIdx.x == 0) part[blockIdx.x] = t;
}
int launch_residual_d(const double2* b, const double2* ax, void* r, bool half, const LatGeo& g, int ls, double scale,
                      double* part, hipStream_t st)
{
  const int64_t n5 = g.stride * ls;
  const int grid = (int)std::min<int64_t>((n5 + 255) / 256, kMaxBlasGrid);
  const bool nt = stream_field(g, ls);
#define QDWF_R(SR, N) \
  hipLaunchKernelGGL((k_residual_d<SR, N>), dim3(grid), dim3(256), 0, st, b, ax, (SpinorIO<SR>::slot_t*)r, ls, n5, scale, part)
  if (half && nt) QDWF_R(Half16, true);
  else if (half) QDWF_R(Half16, false);
  else if (nt) QDWF_R(float, true);
  else QDWF_R(float, false);
#undef QDWF_R
  return grid;
}

// ------------------------------------------------------------------ hop
// acc += the 8 hop terms (without the factor -1/2) of one 5D site.
// load(d, raw) reads neighbour d's spinor, link(i) is element i of the
// site's 72 link entries (LDS).  The spinor of the next direction is
// requested as soon as the current one has been projected to its half
// spinor, so that a wave always has 12 loads in flight while it multiplies
// (acc, the loads and the half spinor are 144 of 168 registers: 3 waves per
// SIMD).  raw holds neighbour 0 already; last(raw) may request
// something else into it behind the last direction's products.
template <bool DAG, class Load, class Link, class Last>
__device__ __forceinline__ void hop_acc_d(Load&& load, Link&& link, Last&& last, double2 raw[12], cplx<double> acc[12])
{
  constexpr int SF = DAG ? 1 : -1, SG = -SF;
#pragma unroll
  for (int k = 0; k < 12; ++k) acc[k] = cmk<double>(0, 0);
#define QDWF_D(D, MU, SGN, NEXT)                                                                        \
  {                                                                                                     \
    cplx<double> w0[3], w1[3];                                                                          \
    _Pragma("unroll") for (int c = 0; c < 3; ++c) proj<MU, SGN>(                                        \
        cmk<double>(raw[c].x, raw[c].y), cmk<double>(raw[3 + c].x, raw[3 + c].y),                       \
        cmk<double>(raw[6 + c].x, raw[6 + c].y), cmk<double>(raw[9 + c].x, raw[9 + c].y), w0[c], w1[c]); \
    if (NEXT >= 0) load(NEXT, raw);                                                                     \
    else last(raw);                                                                                     \
    _Pragma("unroll") for (int r = 0; r < 3; ++r)                                                       \
    {                                                                                                   \
      const cplx<double> u0 = link((D) * 9 + r * 3), u1 = link((D) * 9 + r * 3 + 1),                    \
                         u2 = link((D) * 9 + r * 3 + 2);                                                \
      const cplx<double> y0 = cfma(cfma(cmul(u0, w0[0]), u1, w0[1]), u2, w0[2]);                        \
      const cplx<double> y1 = cfma(cfma(cmul(u0, w1[0]), u1, w1[1]), u2, w1[2]);                        \
      acc[r] = cadd(acc[r], y0);                                                                        \
      acc[3 + r] = cadd(acc[3 + r], y1);                                                                \
      recon_lower<MU, SGN>(y0, y1, acc[6 + r], acc[9 + r]);                                             \
    }                                                                                                   \
  }
  QDWF_D(0, 0, SF, 1) QDWF_D(1, 1, SF, 2) QDWF_D(2, 2, SF, 3) QDWF_D(3, 3, SF, 4)
  QDWF_D(4, 0, SG, 5) QDWF_D(5, 1, SG, 6) QDWF_D(6, 2, SG, 7) QDWF_D(7, 3, SG, -1)
#undef QDWF_D
}

// The block's links (SB sites x 72) and neighbour indices into LDS; the
// caller synchronises.  A thread's NL link loads (NL * blockDim >= 72 SB) are
// all issued before the first goes to LDS.
template <int SB, int NL>
__device__ __forceinline__ void stage_links_d(double2 (*sl)[SB], int (*nbs)[SB], const double2* __restrict__ links,
                                              const LatGeo& g, int64_t h0, int eo_out)
{
  const double2* __restrict__ l = links + lidx(g.stride, eo_out == 2 ? 0 : 1, 0, h0);
  const int bd = blockDim.x, t = threadIdx.x;
  double2 v[NL];
#pragma unroll
  for (int j = 0; j < NL; ++j) {
    const int i = t + j * bd;
    if (i < 72 * SB) v[j] = load_nt(&l[(i / SB) * 64 + (i % SB)]);
  }
  for (int i = t; i < 8 * SB; i += bd) {  // thread (site, d): neighbour d
    const int st = i % SB, d = i / SB;
    if (h0 + st < g.vh) nbs[d][st] = (int)neighbour_of(g, h0 + st, eo_out, d);
  }
#pragma unroll
  for (int j = 0; j < NL; ++j) {
    const int i = t + j * bd;
    if (i < 72 * SB) sl[i / SB][i % SB] = v[j];
  }
}

// out = alpha H in (+ beta_s x): block = SB sites, its waves take the rows
// in turn.  Bound by the traffic beyond the 4 MB L2 of an XCD: the rows of
// the sites in flight on its 32 CUs are larger than that, so a spinor is
// fetched 4.3 times per launch at 24^3x64 Ls12 (0.78 ms, 7.6 TB/s in all), 2.5
// times at 16^3x32 Ls8.  Before the links' loads were batched and the next
// spinor requested early: 0.88 ms, at 16^3x32 Ls8 90 us (now 64), at 8^3x16
// Ls12 28 us (now 7.7).  x is requested behind the last direction's products:
// inside Mpc^+ Mpc 98 against 109 us at 16^3x32 Ls8, 10.2 against 11.8 us at
// 8^3x16 Ls8.
template <int SB, int NW, bool DAG, bool XPAY, bool NT>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(SB == 64 ? 2 : 3))) k_hop_d(HopDArgs a)
{
  __shared__ double2 sl[72][SB];
  __shared__ int nbs[8][SB];
  if (a.cg && a.cg->done) return;
  const int64_t h0 = xcd_logical_block(blockIdx.x, (int64_t)gridDim.x) * SB;
  stage_links_d<SB, (72 * SB + 64 * NW - 1) / (64 * NW)>(sl, nbs, (const double2*)a.links, a.geo, h0, a.eo_out);
  __syncthreads();
  const int site = threadIdx.x % SB;
  const int64_t h = h0 + site;
  if (h >= a.geo.vh) return;
  const double2* __restrict__ in = (const double2*)a.in;
  const double sc = -0.5 * a.alpha;
  for (int s = threadIdx.x / SB; s < a.ls; s += 64 * NW / SB) {
    // the links stay in LDS: read anew for every row (hoisted out of the
    // loop they would take 288 registers)
    asm volatile("" ::: "memory");
    auto load = [&](int d, double2 raw[12]) {
      const double2* __restrict__ p = in + sidx<12>(a.ls, s, 0, nbs[d][site]);
#pragma unroll
      for (int k = 0; k < 12; ++k) raw[k] = p[k * 64];
    };
    cplx<double> acc[12];
    double2 raw[12];
    load(0, raw);
    hop_acc_d<DAG>(
        load,
        [&](int i) {
          const double2 u = sl[i][site];
          return cmk<double>(u.x, u.y);
        },
        [&](double2 xv[12]) {
          if (!XPAY) return;
          const double2* __restrict__ x = (const double2*)a.x + sidx<12>(a.ls, s, 0, h);
#pragma unroll
          for (int k = 0; k < 12; ++k) xv[k] = load_in<NT>(&x[k * 64]);
          __builtin_amdgcn_sched_barrier(0);  // (not to be moved behind the products)
        },
        raw, acc);
    cplx<double> v[12];
#pragma unroll
    for (int k = 0; k < 12; ++k) v[k] = cmk<double>(sc * acc[k].re, sc * acc[k].im);
    if (a.gamma) {  // (D_- only)
      const cplx<double> g = a.gamma[s];
#pragma unroll
      for (int k = 0; k < 12; ++k) v[k] = cmul(g, v[k]);
    }
    if (XPAY) {
      const cplx<double> b = a.beta[s];
#pragma unroll
      for (int k = 0; k < 12; ++k) v[k] = cfma(v[k], b, cmk<double>(raw[k].x, raw[k].y));
    }
    SpinorIO<double>::store_stream((double2*)a.out, a.ls, s, h, v);
  }
}

template <int SB, int NW>
static void launch_hop_d_sb(const HopDArgs& a, bool dag, hipStream_t st)
{
  const dim3 grid((unsigned)((a.geo.vh + SB - 1) / SB));
  const dim3 blk(64 * NW);
  const bool xpay = a.x != nullptr;
  const bool nt = xpay && stream_field(a.geo, a.ls);
  if (!dag && !xpay) hipLaunchKernelGGL((k_hop_d<SB, NW, false, false, false>), grid, blk, 0, st, a);
  if (dag && !xpay) hipLaunchKernelGGL((k_hop_d<SB, NW, true, false, false>), grid, blk, 0, st, a);
  if (!dag && xpay && !nt) hipLaunchKernelGGL((k_hop_d<SB, NW, false, true, false>), grid, blk, 0, st, a);
  if (dag && xpay && !nt) hipLaunchKernelGGL((k_hop_d<SB, NW, true, true, false>), grid, blk, 0, st, a);
  if (!dag && xpay && nt) hipLaunchKernelGGL((k_hop_d<SB, NW, false, true, true>), grid, blk, 0, st, a);
  if (dag && xpay && nt) hipLaunchKernelGGL((k_hop_d<SB, NW, true, true, true>), grid, blk, 0, st, a);
}

void launch_hop_d(const HopDArgs& a, bool dag, hipStream_t st)
{
  // 64 sites: a gather shifted by one site then touches 9 cache lines per KB
  // instead of 12 (24^3x64 Ls12 without z tiles: 0.81 against 0.88 ms; 16^3x32 Ls8: 64
  // against 75 us), but it takes some 200 blocks to fill the chip (10x12^2x20
  // Ls12, 225 blocks: 25.4 against 28.5 us; 8^3x16 Ls12, 64 blocks: 14.1
  // against 7.0 us)
  if (a.geo.vh >= 64 * 200) launch_hop_d_sb<64, 4>(a, dag, st);
  else launch_hop_d_sb<16, 3>(a, dag, st);
}

// out = alpha Mat (H in) (+ beta x), with DOT also the block's part of
// Re <dotp, out>.  Block = SB sites x ls rows (rows up to a multiple of 4):
// thread (site, row) forms the hop of its 5D site, the results go through LDS
// (over the links) one chirality after the other (half the LDS), and the
// waves take the (component, 16 sites) pairs of the s-matrix product in turn.
// Bound like k_hop_d: 0.82 to 0.85 ms at 24^3x64 Ls12 (a spinor fetched 3.7
// times, 6.3 TB/s beyond the L2); 80 us at 16^3x32 Ls8 (97 with the product row
// by row from LDS on the vector units), 11 us at 8^3x16 Ls8.  With x and the
// dot product 117 and 14 us, 108 and 12 us with dotp requested before the
// s-matrix product.
template <int SB, int LSMAX, bool DAG, bool XPAY, bool REAL, bool DOT, bool NT>
__global__ void __launch_bounds__(SB * LSMAX) __attribute__((amdgpu_waves_per_eu(3))) k_hop_m5d(HopM5dArgs a)
{
  typedef SMat<LSMAX, REAL> Mx;
  constexpr int NSLOT = 72 > LSMAX * 6 ? 72 : LSMAX * 6;
  constexpr int ROWS = LSMAX == 8 ? 4 : LSMAX == 12 ? 12 : LSMAX == 16 ? 16 : LSMAX == 24 ? 20 : 28;  // fewest rows
  __shared__ double2 buf[NSLOT][SB];  // links [72][SB], then hop results [LSMAX * 6][SB] of one chirality
  __shared__ int nbs[8][SB];
  if (a.cg && a.cg->done) return;
  const int64_t lb = xcd_logical_block(blockIdx.x, (int64_t)gridDim.x);
  const int64_t h0 = lb * SB;
  stage_links_d<SB, (72 + ROWS - 1) / ROWS>(buf, nbs, a.links, a.geo, h0, a.eo_out);
  __syncthreads();
  const int ls = a.ls;
  const int site = threadIdx.x % SB, row = threadIdx.x / SB;
  cplx<double> acc[12];
  if (h0 + site < a.geo.vh && row < ls) {
    auto load = [&](int d, double2 raw[12]) {
      const double2* __restrict__ p = a.in + sidx<12>(ls, row, 0, nbs[d][site]);
#pragma unroll
      for (int k = 0; k < 12; ++k) raw[k] = p[k * 64];
    };
    double2 raw[12];
    load(0, raw);
    hop_acc_d<DAG>(
        load,
        [&](int i) {
          const double2 u = buf[i][site];
          return cmk<double>(u.x, u.y);
        },
        [](double2*) {}, raw, acc);
  } else {  // (rows beyond ls are operands of the products)
#pragma unroll
    for (int k = 0; k < 12; ++k) acc[k] = cmk<double>(0, 0);
  }
  const double sc = -0.5 * a.alpha;
  const int lane = threadIdx.x & 63, li = lane & 15, lq = lane >> 4;
  const int wv = threadIdx.x >> 6, nw = blockDim.x >> 6, nkb = (ls + 3) >> 2;
  constexpr int UNITS = 6 * SB / 16;  // (component, 16 sites) pairs of a chirality
  double dot = 0.0;
#pragma unroll
  for (int chi = 0; chi < 2; ++chi) {
    Mx m;
    m.load(a.mat + chi * ls * ls, ls);
    __syncthreads();  // every thread is done with the links / the other chirality
#pragma unroll
    for (int k = 0; k < 6; ++k)
      buf[row * 6 + k][site] = make_double2(sc * acc[chi * 6 + k].re, sc * acc[chi * 6 + k].im);
    __syncthreads();
    // the units of both chiralities in turn over the waves
    for (int u = (wv + nw - (chi * UNITS) % nw) % nw; u < UNITS; u += nw) {
      const int k = u / (SB / 16), st = (u % (SB / 16)) * 16 + li;
      const int64_t h = h0 + st;
      const bool act = h < a.geo.vh;
      mf4d dr[Mx::MT], di[Mx::MT];
#pragma unroll
      for (int mt = 0; mt < Mx::MT; ++mt) dr[mt] = di[mt] = (mf4d){0.0, 0.0, 0.0, 0.0};
      constexpr bool EARLY = DOT && Mx::MT == 1;  // (two row tiles have no registers for it)
      double2 xv[Mx::MT][4], pv[Mx::MT][4];
      if (XPAY || EARLY) {
#pragma unroll
        for (int mt = 0; mt < Mx::MT; ++mt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int s = mt * 16 + lq + 4 * i;
            const unsigned o = sidx<12>(ls, s, chi * 6 + k, h);
            if (XPAY && act && s < ls) xv[mt][i] = load_in<NT>(&a.x[o]);
            if (EARLY && act && s < ls) pv[mt][i] = load_in<NT>(&a.dotp[o]);
          }
      }
#pragma unroll
      for (int kb = 0; kb < Mx::KB; ++kb)
        if (kb < nkb) m.fma(kb, buf[(4 * kb + lq) * 6 + k][st], dr, di);
#pragma unroll
      for (int mt = 0; mt < Mx::MT; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int s = mt * 16 + lq + 4 * i;
          if (!act || s >= ls) continue;
          const unsigned o = sidx<12>(ls, s, chi * 6 + k, h);
          double2 v = make_double2(dr[mt][i], di[mt][i]);
          if (XPAY) {
            v.x += a.beta * xv[mt][i].x;
            v.y += a.beta * xv[mt][i].y;
          }
          store_nt(&a.out[o], v);
          if (DOT) {
            const double2 p = EARLY ? pv[mt][i] : load_in<NT>(&a.dotp[o]);
            dot += p.x * v.x + p.y * v.y;
          }
        }
    }
  }
  if (DOT) {
    dot = block_sum<SB * LSMAX / 64>(dot);
    if (threadIdx.x == 0) a.part[lb] = dot;
  }
}

template <int SB, int LSMAX>
static bool launch_hop_m5d_ls(const HopM5dArgs& a, bool dag, hipStream_t st)
{
  const dim3 grid((unsigned)((a.geo.vh + SB - 1) / SB));
  const dim3 blk(SB * ((a.ls + 3) / 4) * 4);
  const bool xpay = a.x != nullptr, dot = a.dotp != nullptr;
  const bool nt = xpay && stream_field(a.geo, a.ls);
#define QDWF_K(D, X, R, DT, N) hipLaunchKernelGGL((k_hop_m5d<SB, LSMAX, D, X, R, DT, N>), grid, blk, 0, st, a)
#define QDWF_L(D, X, DT)                       \
  {                                            \
    if (nt) {                                  \
      if (a.real_mat) QDWF_K(D, X, true, DT, X);  \
      else QDWF_K(D, X, false, DT, X);         \
    } else {                                   \
      if (a.real_mat) QDWF_K(D, X, true, DT, false);  \
      else QDWF_K(D, X, false, DT, false);     \
    }                                          \
    return true;                               \
  }
  if (dag && xpay && dot) QDWF_L(true, true, true)
  if (dot) return false;
  if (!dag && !xpay) QDWF_L(false, false, false)
  if (dag && !xpay) QDWF_L(true, false, false)
  if (dag && xpay) QDWF_L(true, true, false)
#undef QDWF_L
#undef QDWF_K
  return false;
}

// 32 sites for Ls <= 8, where 16 would be blocks of one or two waves, if
// that leaves every CU a block: Mpc^+ Mpc at 16^3x32 Ls8 376 against 389 us,
// 8^3x32 Ls8 (256 blocks) 63 against 67 us; at Ls 12 16 sites are faster
// (8^3x16: 51 against 60 us, 24^3x64: 4.21 against 4.25 ms).
static int hop_m5d_sb(const LatGeo& g, int ls) { return ls <= 8 && g.vh >= 32 * 256 ? 32 : 16; }
int64_t hop_m5d_blocks(const LatGeo& g, int ls) { return (g.vh + hop_m5d_sb(g, ls) - 1) / hop_m5d_sb(g, ls); }

bool launch_hop_m5d(const HopM5dArgs& a, bool dag, hipStream_t st)
{
  if (hop_m5d_sb(a.geo, a.ls) == 32) return launch_hop_m5d_ls<32, 8>(a, dag, st);
  if (a.ls <= 8) return launch_hop_m5d_ls<16, 8>(a, dag, st);
  if (a.ls <= 12) return launch_hop_m5d_ls<16, 12>(a, dag, st);
  if (a.ls <= 16) return launch_hop_m5d_ls<16, 16>(a, dag, st);
  if (a.ls <= 24) return launch_hop_m5d_ls<16, 24>(a, dag, st);
  return launch_hop_m5d_ls<16, 32>(a, dag, st);
}

}  // namespace qdwf
