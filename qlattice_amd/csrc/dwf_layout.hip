// Layout conversion between the reference's array-of-structures complex128
// fields and the blocked device layout (dwf_common.h): 5D fields,
// propagator columns, gauge links.
#include "dwf_internal.h"

namespace qdwf {

// Reference 5D field AoS complex128 [site][s][12] (full, V sites) or
// [half][s][12] (half field) <-> blocked half field of one parity.  `full`
// selects which: for a full field the half-site h of parity eo sits at full
// index of half_coord(h, eo).
// A block converts 16 consecutive device sites x 4 rows through LDS, so that
// both sides of the transpose move whole cache lines: a site's rows are one
// run of 768 bytes in the AoS field, and a (row, component) is 256 bytes of
// its 64-site span in the blocked field.  (With one 16-byte slot per thread
// straight from one side to the other, every 128-byte line of the AoS field
// was requested eight times.)  The source is read with non-temporal loads:
// without them the unpack took 0.62 ms instead of 0.31.
// HBM bound: at 24^3x64 Ls12 (2.04 GB moved) pack 1.32 -> 0.35 ms, unpack
// 2.25 -> 0.31 ms (5.8 and 6.6 TB/s); 16^3x32 Ls8 0.089 and 0.106 -> 0.034 ms.
// Blocks of 64, 32 and 16 sites x 4, 8 and 16 rows were within 7% of each
// other; the smallest leaves small lattices the most blocks.
constexpr int kPackRows = 4;
constexpr int kPackSites = 16;
constexpr int64_t kPackStream = (int64_t)32 << 20;  // bytes of a half field
struct Pack5Args {
  LatGeo geo;
  int ls;
  int full;
  int eo[2];        // parity of blockIdx.y
  double2* soa[2];  // its blocked field
  double2* aos;
};

template <bool PACK, bool NT>
__global__ void __launch_bounds__(256) k_layout5(Pack5Args a)
{
  constexpr int SITES = kPackSites, ROWS = kPackRows;
  // rows padded by one slot: the AoS side walks r at a fixed site
  __shared__ double2 buf[ROWS * 12][SITES + 1];
  __shared__ int64_t run[SITES];  // first AoS element of a site's rows (-1: beyond the field)
  // the row groups of a block's sites back to back on one XCD: together they
  // cover whole sites of the AoS field
  const int nchunk = (a.ls + ROWS - 1) / ROWS;
  const unsigned lb = (unsigned)xcd_logical_block(blockIdx.x, (int64_t)gridDim.x);
  const int64_t h0 = (int64_t)(lb / (unsigned)nchunk) * SITES;
  const int s0 = (int)(lb % (unsigned)nchunk) * ROWS;
  const int nr = (a.ls - s0 < ROWS ? a.ls - s0 : ROWS) * 12;
  if (threadIdx.x < SITES) {
    const int64_t h = h0 + threadIdx.x;
    int64_t r = -1;
    if (h < a.geo.vh) {
      int x[4];
      half_coord(a.geo, h, a.eo[blockIdx.y], x);
      const int64_t site = a.full ? full_index(a.geo, x) : full_index(a.geo, x) / 2;
      r = (site * a.ls + s0) * 12;
    }
    run[threadIdx.x] = r;
  }
  // slot (row r, site) of the block's span
  double2* __restrict__ soa = a.soa[blockIdx.y] + sidx<12>(a.ls, s0, 0, h0);
  constexpr int N = SITES * ROWS * 12 / 256;
  const int site = threadIdx.x % SITES, row = threadIdx.x / SITES;
  constexpr int RS = 256 / SITES;  // rows per pass of the block
  double2 v[N];
  if constexpr (PACK) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int e = threadIdx.x + i * 256, st = e / (ROWS * 12), r = e - st * (ROWS * 12);
      if (r < nr && run[st] >= 0) v[i] = load_in<NT>(&a.aos[run[st] + r]);
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int e = threadIdx.x + i * 256, st = e / (ROWS * 12), r = e - st * (ROWS * 12);
      buf[r][st] = v[i];
    }
    __syncthreads();
    if (run[site] >= 0)
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int r = row + i * RS;
        if (r < nr) soa[r * 64 + site] = buf[r][site];
      }
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int r = row + i * RS;
      if (r < nr) v[i] = load_in<NT>(&soa[r * 64 + site]);
    }
#pragma unroll
    for (int i = 0; i < N; ++i) buf[row + i * RS][site] = v[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int e = threadIdx.x + i * 256, st = e / (ROWS * 12), r = e - st * (ROWS * 12);
      if (r < nr && run[st] >= 0) a.aos[run[st] + r] = buf[r][st];
    }
  }
}

template <bool PACK>
static void launch_layout5(double2* aos, double2* soa0, double2* soa1, const LatGeo& g, int ls, int eo0, int eo1,
                           int full, hipStream_t st)
{
  Pack5Args a;
  a.geo = g;
  a.ls = ls;
  a.full = full;
  a.eo[0] = eo0;
  a.eo[1] = eo1;
  a.soa[0] = soa0;
  a.soa[1] = soa1;
  a.aos = aos;
  const int64_t nblk = (g.vh + kPackSites - 1) / kPackSites * ((ls + kPackRows - 1) / kPackRows);
  const dim3 grid((unsigned)nblk, soa1 ? 2 : 1);
  if (nblk * kPackSites * kPackRows * 192 > kPackStream) hipLaunchKernelGGL((k_layout5<PACK, true>), grid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL((k_layout5<PACK, false>), grid, dim3(256), 0, st, a);
}

void launch_pack5(const double2* aos, double2* soa, const LatGeo& g, int ls, int eo, int full, hipStream_t st)
{
  launch_layout5<true>(const_cast<double2*>(aos), soa, nullptr, g, ls, eo, eo, full, st);
}
void launch_unpack5(const double2* soa, double2* aos, const LatGeo& g, int ls, int eo, int full, hipStream_t st)
{
  launch_layout5<false>(aos, const_cast<double2*>(soa), nullptr, g, ls, eo, eo, full, st);
}
// both parities of a full field in one launch
void launch_pack5_full(const double2* aos, double2* even, double2* odd, const LatGeo& g, int ls, hipStream_t st)
{
  launch_layout5<true>(const_cast<double2*>(aos), even, odd, g, ls, 2, 1, 1, st);
}
void launch_unpack5_full(const double2* even, const double2* odd, double2* aos, const LatGeo& g, int ls,
                         hipStream_t st)
{
  launch_layout5<false>(aos, const_cast<double2*>(even), const_cast<double2*>(odd), g, ls, 2, 1, 1, st);
}

// Propagator column j ([site][12 rows][12 cols] complex128) -> 5D half field
// of parity eo: the chiral embedding of fermion_field_5d_from_4d
// (qcd-prop.h:96-116) with upper = 0, lower = Ls-1 (qcd-prop.h:157):
// spins 0,1 go to s = 0, spins 2,3 to s = Ls-1, everything else is zero.
// With col < 0 the input is a 4D fermion field [site][12].
__global__ void __launch_bounds__(kBlasBlock) k_prop_col_to_5d(const double2* __restrict__ src, double2* __restrict__ soa,
                                                               LatGeo g, int ls, int eo, int col)
{
  const int64_t n = g.vh * ls * 12;
  for (int64_t i = (int64_t)blockIdx.x * kBlasBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlasBlock) {
    const int64_t h = i % g.vh, q = i / g.vh;
    const int s = (int)(q / 12), k = (int)(q - (int64_t)(q / 12) * 12);
    double2 v = make_double2(0.0, 0.0);
    const bool take = (k < 6) ? (s == 0) : (s == ls - 1);
    if (take) {
      int x[4];
      half_coord(g, h, eo, x);
      const int64_t site = full_index(g, x);
      v = (col >= 0) ? src[(site * 12 + k) * 12 + col] : src[site * 12 + k];
    }
    soa[sidx<12>(ls, s, k, h)] = v;
  }
}

// 5D half field of parity eo -> propagator column j (fermion_field_4d_from_5d,
// qcd-prop.h:118-138, upper = Ls-1, lower = 0, qcd-prop.h:164).
__global__ void __launch_bounds__(kBlasBlock) k_5d_to_prop_col(const double2* __restrict__ soa, double2* __restrict__ dst,
                                                               LatGeo g, int ls, int eo, int col)
{
  const int64_t n = g.vh * 12;
  for (int64_t i = (int64_t)blockIdx.x * kBlasBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlasBlock) {
    const int64_t h = i % g.vh;
    const int k = (int)(i / g.vh);
    const int s = (k < 6) ? ls - 1 : 0;
    int x[4];
    half_coord(g, h, eo, x);
    const int64_t site = full_index(g, x);
    const double2 v = soa[sidx<12>(ls, s, k, h)];
    if (col >= 0) dst[(site * 12 + k) * 12 + col] = v;
    else dst[site * 12 + k] = v;
  }
}

void launch_prop_col_to_5d(const double2* src, double2* soa, const LatGeo& g, int ls, int eo, int col, hipStream_t st)
{
  const int64_t n = g.vh * ls * 12;
  hipLaunchKernelGGL(k_prop_col_to_5d, dim3(blas_grid(n)), dim3(kBlasBlock), 0, st, src, soa, g, ls, eo, col);
}
void launch_5d_to_prop_col(const double2* soa, double2* dst, const LatGeo& g, int ls, int eo, int col, hipStream_t st)
{
  const int64_t n = g.vh * 12;
  hipLaunchKernelGGL(k_5d_to_prop_col, dim3(blas_grid(n)), dim3(kBlasBlock), 0, st, soa, dst, g, ls, eo, col);
}

__global__ void __launch_bounds__(kBlasBlock) k_neighbours(unsigned* __restrict__ nbt, LatGeo g)
{
  const int64_t h = (int64_t)blockIdx.x * kBlasBlock + threadIdx.x;
  const int pd = blockIdx.y;  // p * 8 + d
  if (h < g.vh) nbt[pd * g.stride + h] = (unsigned)neighbour_of(g, h, pd < 8 ? 2 : 1, pd & 7);
}
void launch_neighbours(unsigned* nbt, const LatGeo& g, hipStream_t st)
{
  hipLaunchKernelGGL(k_neighbours, dim3((unsigned)((g.vh + kBlasBlock - 1) / kBlasBlock), 16), dim3(kBlasBlock), 0, st,
                     nbt, g);
}

// Gauge AoS [site][mu][3][3] complex128 -> per-output-parity 8-link layout
// (dwf_common.h), FP64 and FP32 copies.  Backward links are stored already
// adjointed: U_mu(x - mu)^+.
__global__ void __launch_bounds__(kBlasBlock) k_pack_gauge(const double2* __restrict__ gauge, double2* __restrict__ l64,
                                                           float2* __restrict__ l32, unsigned* __restrict__ l16,
                                                           LatGeo g)
{
  const int64_t n = g.vh * 2 * 8;
  for (int64_t i = (int64_t)blockIdx.x * kBlasBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlasBlock) {
    const int64_t h = i % g.vh, q = i / g.vh;
    const int p = (int)(q / 8), d = (int)(q % 8);
    const int eo = (p == 0) ? 2 : 1;
    int x[4];
    half_coord(g, h, eo, x);
    const int mu = d & 3;
    if (d >= 4) x[mu] = wrap_dec(x[mu], g.n[mu]);
    const int64_t site = full_index(g, x);
    const double2* U = &gauge[(site * 4 + mu) * 9];
    for (int r = 0; r < 3; ++r)
      for (int c = 0; c < 3; ++c) {
        double2 v = (d < 4) ? U[r * 3 + c] : make_double2(U[c * 3 + r].x, -U[c * 3 + r].y);
        const int64_t off = lidx(g.stride, p, d * 9 + r * 3 + c, h);
        l64[off] = v;
        l32[off] = make_float2((float)v.x, (float)v.y);
        if (l16) l16[off] = pack_h2((float)v.x, (float)v.y);
      }
  }
}

void launch_pack_gauge(const double2* gauge, double2* l64, float2* l32, unsigned* l16, const LatGeo& g,
                       hipStream_t st)
{
  const int64_t n = g.vh * 16;
  hipLaunchKernelGGL(k_pack_gauge, dim3(blas_grid(n)), dim3(kBlasBlock), 0, st, gauge, l64, l32, l16, g);
}

}  // namespace qdwf
