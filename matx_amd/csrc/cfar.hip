// Cell-averaging CFAR: rectangular training window minus a centred guard
// hole, threshold from Pfa (replaces conv2d(xPow, mask, FULL) + trim +
// baTrim/normTrim + calcDets, examples/simple_radar_pipeline.h:394-436,
// 485-492, op body :86-98).
//
// The masked sum is built from positive partial sums only, never as
// "outer box minus hole": a strong target inside the hole would otherwise
// cancel catastrophically in float.  Per input row the kernel forms
//   L = sum of the HX-EX cells left of the hole columns,
//   M = sum over the 2EX+1 hole columns,  Rt = the cells right of them,
// and per output cell
//   sum = sum_{|dy| <= HY, |dy| > EY} (L+M+Rt)(y+dy) + sum_{|dy| <= EY} (L+Rt)(y+dy).
// norm (the count of in-bounds training cells) is exact integer arithmetic,
// ba = sum/norm (IEEE division, as MatX divides), alpha = norm*(pfa^(-1/norm)-1)
// in float as calcDets evaluates it, det = pow > alpha*ba.
//
// Two kernels form the sums alike, bit for bit.  cfar_strip_kernel streams the
// rows of an input with unit column stride through registers and a small LDS
// ring; cfar_kernel takes the rest: other column strides, rows that share
// memory, maps under four columns, windows over four rows either side.
//
// Tiling of cfar_kernel: a one-wave workgroup owns 256 consecutive columns x 16 rows of one
// channel; each lane owns four adjacent columns.  Walking down the rows, a
// lane reads its columns plus the window halo straight from memory (16-byte
// accesses; the overlap between neighbouring lanes is served by the cache,
// so HBM sees each cell about once), forms the horizontal window sums of its
// four columns with shared partial sums, keeps the last 2HY+1 rows in
// registers, and writes each detection row as one 16-byte store.  No LDS
// staging and no barriers: residency is bounded by registers only.
#include <cmath>
#include <type_traits>

#include "fft_engine.hpp"
#include "mxr_cache.hpp"

namespace mxr {

struct CfarArgs {
  const void *in;
  int in_c64;
  int64_t is_c, is_y, is_x;
  int *dets;
  int64_t ds_c, ds_y, ds_x;
  float *ba;
  int64_t bs_c, bs_y, bs_x;
  float *pwo;
  int64_t os_c, os_y, os_x;
  int C, Ny, Nx;
  float pfa;
  int vec_in;    // f32 input, unit column stride, 16-byte aligned rows
  int vec_dets;  // detections: unit column stride, 16-byte aligned rows
  int strip_ok;  // cfar_strip_kernel takes these views
  int unit_out;  // every output: unit column stride
  int strips, bands, band_rows;  // cfar_strip_kernel's split
};

constexpr int CF_NT = 64;             // one wave per workgroup
constexpr int CF_CPL = 4;             // adjacent columns per lane
constexpr int CF_TX = CF_NT * CF_CPL;  // 256 columns per tile
constexpr int CF_TY = 16;             // output rows per tile

// Sums of the four windows u[j .. j+W-1], j = 0..3, sharing partial sums
// (positive terms only, any association is exact up to rounding).
template <int W>
__device__ __forceinline__ void win4(const float *u, float (&o)[4]) {
  if constexpr (W <= 0) {
    o[0] = o[1] = o[2] = o[3] = 0.f;
  } else if constexpr (W == 1) {
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = u[j];
  } else if constexpr (W == 2) {
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = u[j] + u[j + 1];
  } else if constexpr (W == 3) {
    const float p1 = u[1] + u[2], p3 = u[3] + u[4];
    o[0] = u[0] + p1;
    o[1] = p1 + u[3];
    o[2] = u[2] + p3;
    o[3] = p3 + u[5];
  } else {
    float core = u[3];  // u[3 .. W-1] is inside all four windows
#pragma unroll
    for (int i = 4; i < W; ++i) core += u[i];
    const float d = u[1] + u[2], e = u[W] + u[W + 1];
    o[0] = (u[0] + d) + core;
    o[1] = (d + core) + u[W];
    o[2] = (u[2] + core) + e;
    o[3] = (core + e) + u[W + 2];
  }
}

// HY/HX: half window (rows/cols); EY/EX: half guard hole.  CIN: input is
// complex (|.|^2 on load).  EXACT: ba = s/norm (IEEE division, written) and
// det = pow > alpha*ba, MatX's operation order; otherwise det = pow >
// (alpha/norm)*s with alpha/norm tabulated per norm count (the same
// threshold up to a few ulp of float rounding).  WPOW: also write pow.
template <int HY, int HX, int EY, int EX, bool CIN, bool EXACT, bool WPOW>
__global__ __launch_bounds__(CF_NT) void cfar_kernel(CfarArgs a) {
  constexpr int HALO = (HX + 3) & ~3;  // whole quads of halo on each side
  constexpr int NQ = 1 + 2 * HALO / 4; // quads a lane reads per row
  constexpr int NV = 4 * NQ;
  constexpr int LH = CF_TY + 2 * HY;
  constexpr int NCELL = (2 * HY + 1) * (2 * HX + 1);
  constexpr int RING = 2 * HY + 1;
  __shared__ float thr_tab[NCELL + 1];

  const int c = blockIdx.z;
  const int y0 = blockIdx.y * CF_TY;
  const int lane = threadIdx.x;
  const int gx0 = blockIdx.x * CF_TX + CF_CPL * lane;  // first column of this lane
  const int Nx = a.Nx, Ny = a.Ny;

  for (int n = lane; n <= NCELL; n += CF_NT) {
    const float nf = (float)n;
    const float alpha = nf * (powf(a.pfa, -1.0f / nf) - 1.0f);
    thr_tab[n] = EXACT ? alpha : alpha / nf;
  }
  __syncthreads();

  using T = typename std::conditional<CIN, float2, float>::type;
  const T *const in_c = reinterpret_cast<const T *>(a.in) + (int64_t)c * a.is_c;
  const int isy = (int)a.is_y, isx = (int)a.is_x;
  // Row ly of the tile -> the NV values at columns gx0-HALO .. gx0+3+HALO,
  // zero outside the map.  Quads wholly inside a row with unit stride load
  // as one 16-byte access; the few quads crossing the map edge go per cell.
  // Neighbouring lanes' quads overlap and are merged by the cache.
  auto load_row = [&](int ly, float (&u)[NV]) {
    const int gy = y0 - HY + ly;
    if (gy < 0 || gy >= Ny) {
#pragma unroll
      for (int i = 0; i < NV; ++i) u[i] = 0.f;
      return;
    }
    const T *rp = in_c + gy * isy;
#pragma unroll
    for (int qd = 0; qd < NQ; ++qd) {
      const int x = gx0 - HALO + 4 * qd;
      if (!CIN && a.vec_in && x >= 0 && x + 3 < Nx) {
        const float4 z = *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(rp) + x);
        u[4 * qd] = z.x;
        u[4 * qd + 1] = z.y;
        u[4 * qd + 2] = z.z;
        u[4 * qd + 3] = z.w;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int xe = x + e;
          float val = 0.f;
          if (xe >= 0 && xe < Nx) {
            const T z = rp[xe * isx];
            if constexpr (CIN) val = z.x * z.x + z.y * z.y;
            else val = z;
          }
          u[4 * qd + e] = val;
        }
      }
    }
  };

  // in-bounds cell count = ro*co - rh*chh: co/chh per column, ro/rh per row
  int co[CF_CPL], chh[CF_CPL];
  float thr_int[CF_CPL];
#pragma unroll
  for (int j = 0; j < CF_CPL; ++j) {
    const int gx = gx0 + j;
    co[j] = min(gx + HX, Nx - 1) - max(gx - HX, 0) + 1;
    chh[j] = min(gx + EX, Nx - 1) - max(gx - EX, 0) + 1;
    thr_int[j] = thr_tab[min(max((2 * HY + 1) * co[j] - (2 * EY + 1) * chh[j], 0), NCELL)];
  }
  const bool lane_live = gx0 < Nx;
  const bool vec_out = a.vec_dets && gx0 + 3 < Nx;
  const int dsy = (int)a.ds_y, dsx = (int)a.ds_x;
  int *const dets_c = a.dets + (int64_t)c * a.ds_c;

  float full[RING][CF_CPL], lr[RING][CF_CPL], ctr[RING][CF_CPL];
  float ua[NV], ub[NV];  // two rows in flight
  load_row(0, ua);
  if (LH > 1) load_row(1, ub);
#pragma unroll
  for (int ly = 0; ly < LH; ++ly) {
    float u[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) u[i] = (ly & 1) ? ub[i] : ua[i];
    if (ly + 2 < LH) {
      if (ly & 1) load_row(ly + 2, ub);
      else load_row(ly + 2, ua);
    }
    // u[HALO + j + d] is column gx0 + j + d
    float L[4], Mh[4], Rt[4];
    win4<HX - EX>(u + HALO - HX, L);
    win4<2 * EX + 1>(u + HALO - EX, Mh);
    win4<HX - EX>(u + HALO + EX + 1, Rt);
    const int k = ly % RING;
#pragma unroll
    for (int j = 0; j < CF_CPL; ++j) {
      lr[k][j] = L[j] + Rt[j];
      full[k][j] = lr[k][j] + Mh[j];
      ctr[k][j] = u[HALO + j];
    }
    if (ly < 2 * HY) continue;
    const int oy = ly - HY;  // tile row of the cells under test
    const int gy = y0 + oy - HY;
    if (gy >= Ny) break;
    if (!lane_live) continue;
    float thr[CF_CPL];
    int nrm[CF_CPL];
    const bool edge = gy < HY || gy + HY >= Ny;
    const int ro = min(gy + HY, Ny - 1) - max(gy - HY, 0) + 1;
    const int rh = min(gy + EY, Ny - 1) - max(gy - EY, 0) + 1;
#pragma unroll
    for (int j = 0; j < CF_CPL; ++j) {
      nrm[j] = ro * co[j] - rh * chh[j];
      // columns past Nx (never stored) can give a meaningless count: clamp
      // the table index
      thr[j] = edge ? thr_tab[min(max(nrm[j], 0), NCELL)] : thr_int[j];
    }
    int det[CF_CPL];
#pragma unroll
    for (int j = 0; j < CF_CPL; ++j) {
      float s = 0.f;
#pragma unroll
      for (int dy = -HY; dy <= HY; ++dy) {
        const int kk = (oy + dy) % RING;
        const float t = (dy >= -EY && dy <= EY) ? lr[kk][j] : full[kk][j];
        s = dy == -HY ? t : s + t;
      }
      const float p = ctr[oy % RING][j];
      if constexpr (EXACT) {
        const float b = s / (float)nrm[j];
        det[j] = p > thr[j] * b ? 1 : 0;
        if (gx0 + j < Nx)
          a.ba[(int64_t)c * a.bs_c + (int64_t)gy * a.bs_y + (int64_t)(gx0 + j) * a.bs_x] = b;
      } else {
        det[j] = p > thr[j] * s ? 1 : 0;
      }
      if constexpr (WPOW) {
        if (gx0 + j < Nx)
          a.pwo[(int64_t)c * a.os_c + (int64_t)gy * a.os_y + (int64_t)(gx0 + j) * a.os_x] = p;
      }
    }
    int *drow = dets_c + gy * dsy;
    if (vec_out) {
      *reinterpret_cast<int4 *>(drow + gx0) = make_int4(det[0], det[1], det[2], det[3]);
    } else {
#pragma unroll
      for (int j = 0; j < CF_CPL; ++j)
        if (gx0 + j < Nx) drow[(gx0 + j) * dsx] = det[j];
    }
  }
}

// Streaming form for an input with unit column stride (f32 power or c64, rows
// at any alignment).  One wave owns a strip of 256 columns (a quad per lane)
// of one channel and walks down a band of rows.  A lane loads its own quad of
// each row once, RING rows ahead (so a wave keeps RING row loads of 1 KiB in
// flight), parks it in the wave's own LDS ring and reads its neighbours'
// quads from there; the outermost HALO columns on either side only feed the
// others, so a strip emits 256 - 2 HALO columns.  The waves of a workgroup
// share nothing but the threshold table: no barrier in the walk.
//
// Rows go through raw buffer resources that cover the rows the band needs and
// no others: rows above and below the map read as zeros (the CFAR's padding),
// the loads ahead of the band's end fetch nothing, and detections of the
// walk's first and last rows, which belong to no cell of the band, are
// dropped.  So the walk has no per-row tests, and its scalar work (one scalar
// unit serves the CU's four SIMDs) is two additions a row.
//
// Bound by HBM at 8 bytes a cell: 8 x 512 x 28673 cells with the 21 x 7 window
// take 237 us (4.0 TB/s; 184 us at a large copy's rate).  The register-only
// form that rows of this odd length used to take needs 985 us; the LDS-staged
// tiles that 16-byte aligned rows used to take held two workgroups per CU,
// which loaded, summed and stored in turn.  5 x 128 x 4517 c64 cells with
// averages and power: 17 us, 58 us in the register-only form.
constexpr int CS_NT = 256;  // four independent waves
constexpr int CS_NW = CS_NT / 64;
constexpr int CS_BAND = 64;  // output rows per band, at most

// LDS written by one lane of a wave and read by others of the same wave: the
// LDS unit keeps a wave's accesses in order, this keeps the compiler's.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int HY, int HX, int EY, int EX, bool CIN, bool EXACT, bool WPOW>
__global__ __launch_bounds__(CS_NT) __attribute__((amdgpu_waves_per_eu(CIN || EXACT || HY > 3 ? 2 : 4)))
void cfar_strip_kernel(CfarArgs a) {
  constexpr int HALO = (HX + 3) & ~3;  // whole quads of halo on each side
  constexpr int HQ = HALO / 4;
  constexpr int OUT = 256 - 2 * HALO;
  constexpr int NQ = 1 + 2 * HQ;  // quads a lane's windows span
  constexpr int NV = 4 * NQ;
  constexpr int NCELL = (2 * HY + 1) * (2 * HX + 1);
  constexpr int RING = 2 * HY + 1;
  constexpr int NLD = CIN ? 2 : 1;   // 16-byte loads per quad
  constexpr int ESZ = CIN ? 8 : 4;
  // a row of the ring: 64 quads and HQ spare ones on either side, so that the
  // outermost lanes' reads stay inside it (their sums are not used)
  constexpr int RS = 256 + 2 * HALO;
  __shared__ __align__(16) float ring[CS_NW][RING][RS];
  __shared__ float thr_tab[NCELL + 1];

  for (int n = threadIdx.x; n <= NCELL; n += CS_NT) {
    const float nf = (float)n;
    const float alpha = nf * (powf(a.pfa, -1.0f / nf) - 1.0f);
    thr_tab[n] = EXACT ? alpha : alpha / nf;
  }
  __syncthreads();

  const int Nx = a.Nx, Ny = a.Ny;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // wave -> (channel, band, strip), strips fastest: a workgroup's waves are
  // neighbours along the rows and meet in their halo columns
  const uint32_t waves = (uint32_t)a.C * a.bands * a.strips, groups = (waves + CS_NW - 1) / CS_NW;
  if (block_id() >= groups) return;
  const uint32_t g = (uint32_t)xcd_remap(block_id(), groups) * CS_NW + wv;
  if (g >= waves) return;  // no barrier follows
  const int strip = (int)(g % a.strips), gb = (int)(g / a.strips);
  const int band = gb % a.bands, c = gb / a.bands;
  const int y0 = band * a.band_rows;
  const int nrow = min(a.band_rows, Ny - y0);  // output rows of this band
  const int xs = strip * OUT - HALO;           // column of lane 0's quad
  const int gx0 = xs + 4 * lane;
  const bool xedge = xs < 0 || xs + 256 > Nx;  // the strip crosses the map's side

  // input rows ya .. yb - 1 of the map, row y at byte (y - ya) * isb; a lane's
  // column is clamped into the row (Nx >= 4), dx = its own column minus that
  const int ya = max(y0 - HY, 0), yb = min(y0 + nrow + HY, Ny);
  const int isb = (int)a.is_y * ESZ;
  const int xl = min(max(gx0, 0), Nx - 4);
  const int dx = gx0 - xl;
  const buf_rsrc rin = make_rsrc(
      reinterpret_cast<const char *>(a.in) + ((int64_t)c * a.is_c + (int64_t)ya * a.is_y) * ESZ,
      (yb - ya - 1) * isb + Nx * ESZ);
  int vin = (y0 - HY - ya) * isb + xl * ESZ;  // of the next row to load
  float4 pre[RING][NLD];
  auto issue = [&](float4 (&z)[NLD]) {
#pragma unroll
    for (int h = 0; h < NLD; ++h) z[h] = buf_load4(rin, vin + 16 * h);
    vin += isb;
  };

  // in-bounds cell count = ro*co - rh*chh: co/chh per column, ro/rh per row
  int co[4], chh[4], nrm[4];
  float thr[4], nrmf[4];
  auto set_thr = [&](int ro, int rh) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      nrm[j] = ro * co[j] - rh * chh[j];
      nrmf[j] = (float)nrm[j];
      // columns past Nx (never stored) can give a meaningless count
      thr[j] = thr_tab[min(max(nrm[j], 0), NCELL)];
    }
  };
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int gx = gx0 + j;
    co[j] = min(gx + HX, Nx - 1) - max(gx - HX, 0) + 1;
    chh[j] = min(gx + EX, Nx - 1) - max(gx - EX, 0) + 1;
  }
  set_thr(2 * HY + 1, 2 * EY + 1);

  // output rows y0 .. y0 + nrow - 1; an idle lane's offset is past every
  // resource.  The walk's first 2 HY rows have negative offsets.
  constexpr int FAR = 0x40000000;
  const bool live = lane >= HQ && lane < 64 - HQ && gx0 < Nx;
  const bool vec = a.unit_out && !xedge;
  auto out_rsrc = [&](const void *base, int64_t sc, int64_t sy, int64_t sx) {
    return make_rsrc(reinterpret_cast<const char *>(base) + ((int64_t)c * sc + (int64_t)y0 * sy) * 4,
                     ((nrow - 1) * (int)sy + (Nx - 1) * (int)sx + 1) * 4);
  };
  const buf_rsrc rd = out_rsrc(a.dets, a.ds_c, a.ds_y, a.ds_x);
  const buf_rsrc rb = EXACT ? out_rsrc(a.ba, a.bs_c, a.bs_y, a.bs_x) : rd;
  const buf_rsrc rp = WPOW ? out_rsrc(a.pwo, a.os_c, a.os_y, a.os_x) : rd;
  const int dsb = (int)a.ds_y * 4, bsb = (int)a.bs_y * 4, osb = (int)a.os_y * 4;
  int vd = -2 * HY * dsb + gx0 * (int)a.ds_x * 4, vb = -2 * HY * bsb + gx0 * (int)a.bs_x * 4,
      vp = -2 * HY * osb + gx0 * (int)a.os_x * 4;
  if (!live) vd = vb = vp = FAR;
  const int dstep = live ? dsb : 0, bstep = live ? bsb : 0, pstep = live ? osb : 0;

  float full[RING][4], lr[RING][4];
#pragma unroll
  for (int sl = 0; sl < RING; ++sl) {
    issue(pre[sl]);
#pragma unroll
    for (int j = 0; j < 4; ++j) full[sl][j] = lr[sl][j] = 0.f;
  }
  int gy = y0 - 2 * HY;  // row of the cells under test
#pragma unroll 1
  for (int ly0 = 0; ly0 < nrow + 2 * HY; ly0 += RING)
#pragma unroll
    for (int sl = 0; sl < RING; ++sl, ++gy) {
      float q[4];
      if constexpr (CIN) {
        const float4 z0 = pre[sl][0], z1 = pre[sl][NLD - 1];
        q[0] = z0.x * z0.x + z0.y * z0.y;
        q[1] = z0.z * z0.z + z0.w * z0.w;
        q[2] = z1.x * z1.x + z1.y * z1.y;
        q[3] = z1.z * z1.z + z1.w * z1.w;
      } else {
        const float4 z0 = pre[sl][0];
        q[0] = z0.x;
        q[1] = z0.y;
        q[2] = z0.z;
        q[3] = z0.w;
      }
      issue(pre[sl]);
      if (xedge) {  // own column j is loaded element j + dx, zero when there is none
        const float o[8] = {q[0], q[1], q[2], q[3], 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; ++j)
          q[j] = dx == 0 ? o[j] : (dx == 1 ? o[j + 1] : (dx == 2 ? o[j + 2] : (dx == 3 ? o[j + 3] : 0.f)));
      }
      // the slot's readers of RING rows ago are this wave's own, in order
      float *row = &ring[wv][sl][4 * lane];
      *reinterpret_cast<float4 *>(row + HALO) = make_float4(q[0], q[1], q[2], q[3]);
      wave_lds_order();
      float u[NV];
#pragma unroll
      for (int m = 0; m < NQ; ++m) {
        if (m == HQ) {
#pragma unroll
          for (int j = 0; j < 4; ++j) u[4 * m + j] = q[j];
          continue;
        }
        const float4 z = *reinterpret_cast<const float4 *>(row + 4 * m);
        u[4 * m] = z.x;
        u[4 * m + 1] = z.y;
        u[4 * m + 2] = z.z;
        u[4 * m + 3] = z.w;
      }
      // u[HALO + j + d] is column gx0 + j + d
      float L[4], Mh[4], Rt[4];
      win4<HX - EX>(u + HALO - HX, L);
      win4<2 * EX + 1>(u + HALO - EX, Mh);
      win4<HX - EX>(u + HALO + EX + 1, Rt);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        lr[sl][j] = L[j] + Rt[j];
        full[sl][j] = lr[sl][j] + Mh[j];
      }
      // rows whose window leaves the map have fewer cells; the row after them
      // goes back to the interior count
      if (gy <= HY || gy + HY >= Ny)
        set_thr(min(gy + HY, Ny - 1) - max(gy - HY, 0) + 1, min(gy + EY, Ny - 1) - max(gy - EY, 0) + 1);
      const float4 cut =
          *reinterpret_cast<const float4 *>(&ring[wv][(sl - HY + RING) % RING][4 * lane + HALO]);
      const float cv[4] = {cut.x, cut.y, cut.z, cut.w};
      int det[4];
      float bav[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float sm = 0.f;
#pragma unroll
        for (int dy = -HY; dy <= HY; ++dy) {
          const int kk = (sl - HY + dy + 2 * RING) % RING;  // ring slot of row ly - HY + dy
          const float t = (dy >= -EY && dy <= EY) ? lr[kk][j] : full[kk][j];
          sm = dy == -HY ? t : sm + t;
        }
        if constexpr (EXACT) {
          bav[j] = sm / nrmf[j];
          det[j] = cv[j] > thr[j] * bav[j] ? 1 : 0;
        } else {
          det[j] = cv[j] > thr[j] * sm ? 1 : 0;
        }
      }
      wave_lds_order();  // the next rows' writes stay behind these reads
      if (vec) {
        buf_store4(rd, vd, make_float4(__int_as_float(det[0]), __int_as_float(det[1]),
                                       __int_as_float(det[2]), __int_as_float(det[3])));
        if constexpr (EXACT) buf_store4(rb, vb, make_float4(bav[0], bav[1], bav[2], bav[3]));
        if constexpr (WPOW) buf_store4(rp, vp, cut);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const bool in = gx0 + j < Nx;
          buf_store1(rd, in ? vd + j * (int)a.ds_x * 4 : FAR, __int_as_float(det[j]));
          if constexpr (EXACT) buf_store1(rb, in ? vb + j * (int)a.bs_x * 4 : FAR, bav[j]);
          if constexpr (WPOW) buf_store1(rp, in ? vp + j * (int)a.os_x * 4 : FAR, cv[j]);
        }
      }
      vd += dstep;
      if constexpr (EXACT) vb += bstep;
      if constexpr (WPOW) vp += pstep;
    }
}

template <int HY, int HX, int EY, int EX, bool CIN, bool EXACT, bool WPOW>
static void launch_cfar3(const CfarArgs &a, dim3 grid, hipStream_t s) {
  cfar_kernel<HY, HX, EY, EX, CIN, EXACT, WPOW><<<grid, dim3(CF_NT), 0, s>>>(a);
}

template <int HY, int HX, int EY, int EX>
static mxr_status launch_cfar(CfarArgs a, hipStream_t s) {
  static_assert(HX <= 16 && HY <= 10, "window");
  const bool ex = a.ba != nullptr, wp = a.pwo != nullptr;
  if constexpr (HY <= 4) {
    if (a.strip_ok) {
      constexpr int OUT = 256 - 2 * ((HX + 3) & ~3);
      a.strips = (a.Nx + OUT - 1) / OUT;
      // rows per band: a band re-reads 2 HY rows of its neighbours, so bands
      // are long (64 rows) where the map still gives every SIMD a few waves,
      // and short on small maps
      a.band_rows = CS_BAND;
      auto waves = [&] { return (int64_t)a.C * a.strips * ((a.Ny + a.band_rows - 1) / a.band_rows); };
      while (a.band_rows > 8 && waves() < 16 * (int64_t)cu_count()) a.band_rows /= 2;
      a.bands = (a.Ny + a.band_rows - 1) / a.band_rows;
      const int64_t G = (waves() + CS_NW - 1) / CS_NW;
      MXR_REQUIRE(G * CS_NW < (1ll << 31), MXR_INVALID_SIZE, "cfar: too many tiles");
      const dim3 grid = linear_grid(G);
      ProfScope ps("cfar_strip_kernel", s);
      auto go = [&]<bool CIN>() {
        if (ex) wp ? cfar_strip_kernel<HY, HX, EY, EX, CIN, true, true><<<grid, dim3(CS_NT), 0, s>>>(a)
                   : cfar_strip_kernel<HY, HX, EY, EX, CIN, true, false><<<grid, dim3(CS_NT), 0, s>>>(a);
        else wp ? cfar_strip_kernel<HY, HX, EY, EX, CIN, false, true><<<grid, dim3(CS_NT), 0, s>>>(a)
                : cfar_strip_kernel<HY, HX, EY, EX, CIN, false, false><<<grid, dim3(CS_NT), 0, s>>>(a);
      };
      if (a.in_c64) go.template operator()<true>();
      else go.template operator()<false>();
      MXR_HIP_TRY(hipGetLastError());
      return MXR_SUCCESS;
    }
  }
  dim3 grid((a.Nx + CF_TX - 1) / CF_TX, (a.Ny + CF_TY - 1) / CF_TY, a.C);
  {
    ProfScope ps("cfar_kernel", s);
    if (a.in_c64) {
      if (ex) wp ? launch_cfar3<HY, HX, EY, EX, true, true, true>(a, grid, s)
              : launch_cfar3<HY, HX, EY, EX, true, true, false>(a, grid, s);
      else wp ? launch_cfar3<HY, HX, EY, EX, true, false, true>(a, grid, s)
              : launch_cfar3<HY, HX, EY, EX, true, false, false>(a, grid, s);
    } else {
      if (ex) wp ? launch_cfar3<HY, HX, EY, EX, false, true, true>(a, grid, s)
              : launch_cfar3<HY, HX, EY, EX, false, true, false>(a, grid, s);
      else wp ? launch_cfar3<HY, HX, EY, EX, false, false, true>(a, grid, s)
              : launch_cfar3<HY, HX, EY, EX, false, false, false>(a, grid, s);
    }
  }
  MXR_HIP_TRY(hipGetLastError());
  return MXR_SUCCESS;
}

mxr_status cfar_impl(const mxr_tensor *dets, const mxr_tensor *ba_out, const mxr_tensor *pow_out,
                     const mxr_tensor *in, const mxr_cfar_params *pp, hipStream_t stream) {
  mxr_status st;
  MXR_REQUIRE(pp != nullptr, MXR_INVALID_PARAMETER, "cfar: null params");
  if ((st = check_tensor(in, "cfar input", 0, 3, 3))) return st;
  MXR_REQUIRE(in->dtype == MXR_F32 || in->dtype == MXR_C64, MXR_INVALID_TYPE,
              "cfar: input must be f32 power or c64");
  if ((st = check_tensor(dets, "cfar detections", MXR_I32, 3, 3))) return st;
  if (ba_out && (st = check_tensor(ba_out, "cfar ba", MXR_F32, 3, 3))) return st;
  if (pow_out && (st = check_tensor(pow_out, "cfar power", MXR_F32, 3, 3))) return st;
  const int64_t C = in->shape[0], Ny = in->shape[1], Nx = in->shape[2];
  for (const mxr_tensor *o : {dets, ba_out, pow_out}) {
    if (!o) continue;
    MXR_REQUIRE(o->shape[0] == C && o->shape[1] == Ny && o->shape[2] == Nx, MXR_INVALID_SIZE,
                "cfar: outputs must match the input shape");
    MXR_REQUIRE(!views_overlap(*o, *in), MXR_ALIAS_ERROR, "cfar: an output aliases the input");
  }
  const int wy = pp->win_y, wx = pp->win_x, gy = pp->guard_y, gx = pp->guard_x;
  MXR_REQUIRE(wy >= 1 && wx >= 1 && (wy & 1) && (wx & 1), MXR_INVALID_PARAMETER,
              "cfar: window %dx%d must have odd positive sides", wy, wx);
  MXR_REQUIRE(gy >= 1 && gx >= 1 && (gy & 1) && (gx & 1) && gy <= wy && gx <= wx,
              MXR_INVALID_PARAMETER, "cfar: guard %dx%d must be odd and inside the window", gy, gx);
  MXR_REQUIRE(pp->pfa > 0.f && pp->pfa < 1.f, MXR_INVALID_PARAMETER, "cfar: pfa must be in (0,1)");
  if (C == 0 || Ny == 0 || Nx == 0) return MXR_SUCCESS;
  MXR_REQUIRE(C <= 65535 && Ny < (1 << 30) && Nx < (1 << 30), MXR_INVALID_SIZE,
              "cfar: shape too large");
  auto chan_span = [&](const mxr_tensor *t) {
    return std::llabs(t->stride[1]) * (Ny - 1) + std::llabs(t->stride[2]) * (Nx - 1);
  };
  MXR_REQUIRE(chan_span(in) < (1ll << 31) && chan_span(dets) < (1ll << 31), MXR_INVALID_SIZE,
              "cfar: one channel of the input or detections spans more than 2^31 elements");
  CfarArgs a{};
  a.in = in->data;
  a.in_c64 = in->dtype == MXR_C64;
  a.is_c = in->stride[0];
  a.is_y = in->stride[1];
  a.is_x = in->stride[2];
  a.dets = (int *)dets->data;
  a.ds_c = dets->stride[0];
  a.ds_y = dets->stride[1];
  a.ds_x = dets->stride[2];
  if (ba_out) {
    a.ba = (float *)ba_out->data;
    a.bs_c = ba_out->stride[0];
    a.bs_y = ba_out->stride[1];
    a.bs_x = ba_out->stride[2];
  }
  if (pow_out) {
    a.pwo = (float *)pow_out->data;
    a.os_c = pow_out->stride[0];
    a.os_y = pow_out->stride[1];
    a.os_x = pow_out->stride[2];
  }
  a.C = (int)C;
  a.Ny = (int)Ny;
  a.Nx = (int)Nx;
  a.pfa = pp->pfa;
  auto aligned16 = [](const mxr_tensor *t) {
    return ((uintptr_t)t->data % 16 == 0) && t->stride[2] == 1 && t->stride[1] % 4 == 0 &&
           t->stride[0] % 4 == 0;
  };
  a.vec_in = in->dtype == MXR_F32 && aligned16(in);
  a.vec_dets = aligned16(dets);
  auto unit = [](const mxr_tensor *t) { return !t || t->stride[2] == 1; };
  a.unit_out = unit(dets) && unit(ba_out) && unit(pow_out);
  if (Ny == 1) a.is_y = Nx, a.ds_y = Nx * a.ds_x, a.bs_y = Nx * a.bs_x, a.os_y = Nx * a.os_x;
  // the streaming kernel addresses the rows of one band (at most CS_BAND
  // output rows, 2 x 4 halo rows and two steps of the walk) with byte offsets
  // below 2^30 from the band's first row, and counts on rows that follow one
  // another in memory: an offset before the first or past the last row is
  // then outside the resource
  auto band_ok = [&](const mxr_tensor *t, int64_t sy, int64_t sx, int64_t esz) {
    return !t || (sx >= 1 && sy >= (Nx - 1) * sx + 1 && ((CS_BAND + 32) * sy + 256 * sx) * esz < (1ll << 30));
  };
  a.strip_ok = unit(in) && Nx >= 4 && band_ok(in, a.is_y, 1, a.in_c64 ? 8 : 4) &&
               band_ok(dets, a.ds_y, a.ds_x, 4) && band_ok(ba_out, a.bs_y, a.bs_x, 4) &&
               band_ok(pow_out, a.os_y, a.os_x, 4);
  const int hy = wy / 2, hx = wx / 2, ey = gy / 2, ex = gx / 2;
#define MXR_CFAR_CASE(HY_, HX_, EY_, EX_) \
  if (hy == HY_ && hx == HX_ && ey == EY_ && ex == EX_) return launch_cfar<HY_, HX_, EY_, EX_>(a, stream);
  MXR_CFAR_CASE(2, 6, 1, 1)   // 5 x 13 window, 3 x 3 hole (MatX mask)
  MXR_CFAR_CASE(2, 6, 1, 2)   // 5 x 13 window, 3 x 5 hole
  MXR_CFAR_CASE(2, 6, 0, 0)
  MXR_CFAR_CASE(1, 1, 0, 0)
  MXR_CFAR_CASE(1, 2, 0, 1)
  MXR_CFAR_CASE(2, 2, 1, 1)
  MXR_CFAR_CASE(2, 4, 1, 1)
  MXR_CFAR_CASE(3, 3, 1, 1)
  MXR_CFAR_CASE(3, 10, 1, 2)  // 7 x 21 window, 3 x 5 hole
  MXR_CFAR_CASE(3, 10, 1, 1)
  MXR_CFAR_CASE(10, 3, 2, 1)  // 21 x 7 window, 5 x 3 hole
  MXR_CFAR_CASE(4, 8, 1, 1)
#undef MXR_CFAR_CASE
  set_error(MXR_NOT_SUPPORTED,
            "cfar: window %dx%d / guard %dx%d has no fused kernel instance (use conv2d + "
            "threshold)", wy, wx, gy, gx);
  return MXR_NOT_SUPPORTED;
}

}  // namespace mxr

extern "C" mxr_status mxr_cfar(const mxr_tensor *dets, const mxr_tensor *ba_out,
                               const mxr_tensor *pow_out, const mxr_tensor *in,
                               const mxr_cfar_params *params, hipStream_t stream) {
  return mxr::guarded("mxr_cfar",
                      [&] { return mxr::cfar_impl(dets, ba_out, pow_out, in, params, stream); });
}
