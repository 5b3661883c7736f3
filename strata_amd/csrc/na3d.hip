// NA3D forward for gfx950.
//
// Semantics follow NATTEN's na3d (0.21.5): clamped windows, optional dilation,
// non-causal, softmax over kz*ky*kx keys scaled by `scale`.  Three kernels:
//
//  * na3d_scalar_kernel: one thread per (batch, query, head), fp32 math, for
//    shapes neither the MFMA kernels nor (fp32 inputs) na3d_gather.hip cover.
//  * na3d_mfma_kernel:   bf16 inputs, fp32 accumulation.  A workgroup owns a
//    (1, NTY*TY, 4*TX) box of queries of one (batch, head, dilation residue);
//    each of its 4 waves owns NTY tiles of (TY, TX) = 16 queries stacked in y.
//    The union of the box's windows streams from HBM straight into an LDS ring
//    (buffer_load ... lds), two (z, y) key rows per stage.  Per stage a wave
//    reads its 16-key K block and the V^T operands once and, for every tile
//    whose windows reach those rows, computes S^T = K Q^T on
//    v_mfma_f32_16x16x32_bf16 (keys on M, queries on N), masks the window,
//    runs an online softmax with lazy rescaling, and accumulates
//    O^T += V^T P^T (V^T via ds_read_b64_tr_b16) and the row sums (ones x P^T)
//    on the same MFMA.
//  * na3d_strip_kernel:  the same tile math for 4-column tiles (kx 10..13,
//    head_dim 64), but a workgroup walks a whole column of tiles along y and
//    streams every key row once, four tiles in flight per wave.
#include <cstdlib>
#include <type_traits>
#include <utility>

#include "common.h"
#include "na3d_gather.h"

namespace strata {

struct Na3dParams {
  const void* q;
  const void* k;
  const void* v;
  void* o;
  int B, H, D;
  int L[3];
  int org[3];
  int ext[3];
  int ker[3];
  int dil[3];
  float scale;
  int64_t qs[5], ks[5], vs[5], os[5];
  float* lse;  // [B, ext0, lse_ext1, ext2, H] log2-sum-exp of the log2-unit scores, or null
  int lse_ext1;  // y extent of the lse array: the caller's box, also for a y sub-box (lse then shifted)
  // Rotary embedding of the queries inside the kernel (head_dim 64, half layout:
  // pair j = (j, j + 32)), or rc == null: fp32 cos / sin tables [B, rzt, L1, L2, 32]
  // indexed by each query's full-grid position, rzt = 1 or L0.
  const float* rc;
  const float* rs;
  int rzt;
};

// Row of the query-RoPE tables for the full-grid position (b, z, y, x).
__device__ __forceinline__ int64_t rope_row(const Na3dParams& p, int b, int z, int y, int x) {
  return (((int64_t)b * p.rzt + (p.rzt == 1 ? 0 : z)) * p.L[1] + y) * p.L[2] + x;
}

// Rotate one lane's query pairs: lo holds dims j0 .. j0 + 7, hi dims j0 + 32 .. j0 + 39
// (pairs j0 .. j0 + 7 of the half layout), c / s their cos / sin; each rotated value
// is rounded to bf16 as the RoPE pack rounds q (rope_pack.hip, rot8).
__device__ __forceinline__ void rope_q_pairs(bf16x8& lo, bf16x8& hi, const float* c, const float* s) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float a = (float)lo[e], b = (float)hi[e];
    lo[e] = (bf16)rope_rot_a(a, b, c[e], s[e]);
    hi[e] = (bf16)rope_rot_b(a, b, c[e], s[e]);
  }
}

// Index of query (box coordinates ez, ey, ex) in the lse output.
__device__ __forceinline__ int64_t lse_index(const Na3dParams& p, int b, int ez, int ey, int ex, int h) {
  return ((((int64_t)b * p.ext[0] + ez) * p.lse_ext1 + ey) * p.ext[2] + ex) * p.H + h;
}

// ---------------------------------------------------------------------------
// Scalar kernel
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ float ld_elem(const T* p) {
  return (float)(*p);
}

template <typename T, int D>
__global__ __launch_bounds__(256) void na3d_scalar_kernel(Na3dParams p, int64_t total) {
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const int h = (int)(idx % p.H);
  int64_t r = idx / p.H;
  const int ex = (int)(r % p.ext[2]);
  r /= p.ext[2];
  const int ey = (int)(r % p.ext[1]);
  r /= p.ext[1];
  const int ez = (int)(r % p.ext[0]);
  const int b = (int)(r / p.ext[0]);

  const int qc[3] = {p.org[0] + ez, p.org[1] + ey, p.org[2] + ex};
  int base[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int d = p.dil[a];
    const int g = qc[a] % d;
    const int Lg = sub_len(p.L[a], g, d);
    base[a] = g + d * win_start(qc[a] / d, Lg, p.ker[a]);
  }

  const T* qp = (const T*)p.q + b * p.qs[0] + qc[0] * p.qs[1] + qc[1] * p.qs[2] + qc[2] * p.qs[3] + h * p.qs[4];
  float qv[D];
#pragma unroll
  for (int d = 0; d < D; ++d) qv[d] = ld_elem(qp + d) * p.scale;

  float acc[D];
#pragma unroll
  for (int d = 0; d < D; ++d) acc[d] = 0.f;
  float m = -INFINITY, l = 0.f;

  const T* kb = (const T*)p.k + b * p.ks[0] + h * p.ks[4];
  const T* vb = (const T*)p.v + b * p.vs[0] + h * p.vs[4];
  for (int jz = 0; jz < p.ker[0]; ++jz) {
    const int z = base[0] + jz * p.dil[0];
    for (int jy = 0; jy < p.ker[1]; ++jy) {
      const int y = base[1] + jy * p.dil[1];
      for (int jx = 0; jx < p.ker[2]; ++jx) {
        const int x = base[2] + jx * p.dil[2];
        const T* kp = kb + z * p.ks[1] + y * p.ks[2] + x * p.ks[3];
        float s = 0.f;
#pragma unroll
        for (int d = 0; d < D; ++d) s = fmaf(qv[d], ld_elem(kp + d), s);
        const float mn = fmaxf(m, s);
        const float alpha = expf(m - mn);
        const float e = expf(s - mn);
        l = l * alpha + e;
        const T* vp = vb + z * p.vs[1] + y * p.vs[2] + x * p.vs[3];
#pragma unroll
        for (int d = 0; d < D; ++d) acc[d] = fmaf(acc[d], alpha, e * ld_elem(vp + d));
        m = mn;
      }
    }
  }
  const float inv = 1.f / l;
  T* op = (T*)p.o + b * p.os[0] + ez * p.os[1] + ey * p.os[2] + ex * p.os[3] + h * p.os[4];
#pragma unroll
  for (int d = 0; d < D; ++d) op[d] = (T)(acc[d] * inv);
  if (p.lse) p.lse[idx] = (m + logf(l)) * 1.4426950408889634f;  // idx enumerates (b, ez, ey, ex, h)
}

// ---------------------------------------------------------------------------
// MFMA kernel
// ---------------------------------------------------------------------------
// Tile bookkeeping shared by host and device.
struct Na3dTiles {
  int nxt, nyt, nzt;  // workgroup tiles per axis (max over residue classes)
  int nres;           // dil_z * dil_y * dil_x
  int total;          // workgroups in the launch
};

// Tile (z, y, x) of the w-th workgroup of one (batch, head, residue class):
// 4 x 4 x 4 blocks of tiles (smaller at the grid's far edges), x fastest
// inside a block.  The ~64 workgroups an XCD runs at once then cover one
// compact block whose z and x/y halos overlap, so the overlapping key rows
// are read from HBM once and from L2 by the neighbours.
__device__ __forceinline__ void blocked_tile(int w, int nz, int ny, int nx, int& z, int& y, int& x) {
  constexpr int BZ = 4, BY = 4, BX = 4;
  const int zb = w / (BZ * ny * nx);
  int r = w - zb * BZ * ny * nx;
  const int bz = min(BZ, nz - zb * BZ);
  const int yb = r / (bz * BY * nx);
  r -= yb * bz * BY * nx;
  const int by = min(BY, ny - yb * BY);
  const int xb = r / (bz * by * BX);
  r -= xb * bz * by * BX;
  const int bx = min(BX, nx - xb * BX);
  x = xb * BX + r % bx;
  r /= bx;
  y = yb * BY + r % by;
  z = zb * BZ + r / by;
}

// Swizzle of the 16-byte chunks of one key row (D bf16 = D/8 chunks) in LDS:
// logical chunk c of key `key` sits at slot c ^ f(key).  f is chosen by
// measurement (SQ_LDS_BANK_CONFLICT of the exact K ds_read_b128 and V
// ds_read_b64_tr_b16 address streams of the kernel, every window offset):
//   D = 32: f = (key >> 1) & 3,  D = 64: f = key & 7,  D = 128: f = (key & 7) << 1
// -- no conflicts on either read for any window offset.
template <int D>
__device__ __forceinline__ int swz(int chunk, int key) {
  if constexpr (D == 32) return chunk ^ ((key >> 1) & 3);
  else if constexpr (D == 64) return chunk ^ (key & 7);
  else return chunk ^ ((key & 7) << 1);
}


// Cross-lane max over lanes l, l^16 and l^32 (the four lanes of one MFMA
// output column) with the gfx950 permlane swaps.
__device__ __forceinline__ float colmax(float x) {
  const uint32_t u = __float_as_uint(x);
  auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const uint32_t v = __float_as_uint(x);
  auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}


constexpr int NA3D_NWX = 4;          // waves per workgroup, side by side along x

// Sum over lanes l, l^16, l^32 (the four lanes of one MFMA output column).
__device__ __forceinline__ float colsum(float x) {
  const uint32_t u = __float_as_uint(x);
  auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const uint32_t v = __float_as_uint(x);
  auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Bits [lo, hi) of a 32-bit mask (empty if hi <= lo).
__device__ __forceinline__ uint32_t bit_range(int lo, int hi) {
  lo = lo < 0 ? 0 : lo;
  hi = hi > 32 ? 32 : hi;
  if (hi <= lo) return 0;
  const uint32_t top = hi == 32 ? ~0u : ((1u << hi) - 1);
  return top & ~((1u << lo) - 1);
}

// Workgroup = 4 waves along x; each wave owns NTY query tiles of (TY, TX) =
// 16 queries stacked along y, so a workgroup covers (1, NTY*TY, 4*TX) queries
// of one (batch, head, dilation residue, z).  K and V rows of the union of
// the workgroup's windows stream through an NBUF-deep LDS ring, two (z, y)
// rows ("a pair") per stage, loaded straight from HBM into LDS.  Each stage's
// K block (16 keys per row) and V^T operands are read from LDS once per wave
// and shared by every tile whose window union covers the pair.
//
// Softmax: scores live in log2 units, u = s*scale*log2(e) - m, where m is a
// per-query reference that starts at the query's score against its own key
// (always inside its window) and only moves up, lazily, when a stage's
// maximum exceeds it by more than TAU.  Q is pre-scaled by scale*log2(e) and
// the QK MFMA starts from C = bias - m (bias in {0, -inf} per key for the x
// mask), so the MFMA itself returns u and no VALU work sits between the scores
// and the exponentials outside the boundary rows of the y mask.
// LDS bytes of one workgroup of the general kernel: a ring of NBUF stages.
template <int D, int TX, int RPS, int NBUF>
constexpr int mfma_lds_bytes() {
  return NBUF * 2 * RPS * (((NA3D_NWX - 1) * TX + 16 + 512 / D - 1) / (512 / D) * (512 / D)) * D * 2;
}

// `lds`: the workgroup's LDS (mfma_lds_bytes), 1 KiB aligned; `id`: its tile
// index in [0, tg.total) (the kernels pass their workgroup id; the fused
// small-window kernel an offset one, in a block of ids starting at a multiple of 8).
// ROPE: rotate the queries (p.rc / p.rs tables; head_dim 64, half layout).
template <int D, int TX, int NTY, int RPS, int NBUF, bool ROPE = false>
__device__ __forceinline__ void na3d_mfma_body(const Na3dParams p, const Na3dTiles tg, char* lds, int id) {
#if defined(__HIP_DEVICE_COMPILE__)  // the body is device code only; the host pass needs just the signature
  constexpr int NWX = NA3D_NWX;
  constexpr int TY = 16 / TX;
  constexpr int WY = NTY * TY;            // workgroup query rows
  constexpr int WQX = NWX * TX;           // workgroup query columns
  constexpr int LW = (NWX - 1) * TX + 16; // keys per LDS row that are read
  constexpr int KPK = 512 / D;            // keys per KiB
  constexpr int LWP = (LW + KPK - 1) / KPK * KPK;
  constexpr int RB = LWP * D * 2;         // bytes per (tensor, row) region
  constexpr int RKB = RB / 1024;
  constexpr int STAGE_B = 2 * RPS * RB;   // K rows 0..RPS-1, then V rows 0..RPS-1
  constexpr int LPT = 2 * RPS * RKB / NWX;  // 1-KiB DMA loads per wave per stage
  constexpr int NRP = RPS / 2;            // row pairs per stage (one PV MFMA k-step each)
  constexpr int CPK = D / 8;              // 16-byte chunks per key
  constexpr int KS = D / 32;              // k-steps of the QK MFMA
  constexpr int DB = D / 16;              // d-blocks of the PV MFMA
  // Lazy-rescale slack (log2 units): probabilities reach at most 2^TAU and the
  // fp32 sums at most |W| * 2^TAU * max|v|, far inside fp32/bf16 range; terms
  // more than 126 below the reference underflow, i.e. are < 2^-126 of the max.
  constexpr float TAU = 64.f;
  static_assert(RB % 1024 == 0 && (2 * RPS * RKB) % NWX == 0 && (RPS == 2 || RPS == 4), "stage layout");

  static_assert(NBUF * STAGE_B == mfma_lds_bytes<D, TX, RPS, NBUF>(), "LDS size");

  const int wg = xcd_tile_order(tg.total, id);
  const int per = tg.nxt * tg.nyt * tg.nzt;
  int t = wg / per;
  int zt, yt, xt;
  blocked_tile(wg - t * per, tg.nzt, tg.nyt, tg.nxt, zt, yt, xt);
  const int res = t % tg.nres;
  t /= tg.nres;
  const int h = t % p.H;
  const int b = t / p.H;
  const int dz = p.dil[0], dy = p.dil[1], dx = p.dil[2];
  const int gx = res % dx;
  const int gy = (res / dx) % dy;
  const int gz = res / (dx * dy);

  const int Lz = sub_len(p.L[0], gz, dz);
  const int Ly = sub_len(p.L[1], gy, dy);
  const int Lx = sub_len(p.L[2], gx, dx);
  const int qz0 = sub_first(p.org[0], gz, dz), qz1 = sub_end(p.org[0], p.ext[0], gz, dz);
  const int qy0 = sub_first(p.org[1], gy, dy), qy1 = sub_end(p.org[1], p.ext[1], gy, dy);
  const int qx0 = sub_first(p.org[2], gx, dx), qx1 = sub_end(p.org[2], p.ext[2], gx, dx);
  const int iz = qz0 + zt;
  const int y0 = qy0 + yt * WY;
  const int x0 = qx0 + xt * WQX;
  if (iz >= qz1 || y0 >= qy1 || x0 >= qx1) return;  // uniform over the workgroup

  const int kz = p.ker[0], ky = p.ker[1], kx = p.ker[2];
  const int sz = win_start(iz, Lz, kz);
  const int Y0 = win_start(y0, Ly, ky);
  const int NR = win_start(min(y0 + WY - 1, qy1 - 1), Ly, ky) + ky - Y0;  // rows of the y-union (<= 64)
  const int NQ = (NR + RPS - 1) / RPS;                                   // stages per z-slice (<= 32)
  const int X0 = win_start(x0, Lx, kx);
  const int nstage = kz * NQ;

  const int tid = (int)__builtin_amdgcn_workitem_id_x();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: keeps DMA descriptors in SGPRs
  const int lane = tid & 63;
  const int n16 = lane & 15;
  const int g = lane >> 4;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;

  // ---- per-lane x geometry (shared by the wave's tiles) ----
  const int xw0 = x0 + wave * TX;
  const int off_w = win_start(min(xw0, qx1 - 1), Lx, kx) - X0;
  const int qx = xw0 + n16 % TX;
  const int qxc = min(qx, qx1 - 1);
  const int sx = win_start(qxc, Lx, kx);
  float xbias[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int kxs = X0 + off_w + 4 * g + i;
    xbias[i] = (kxs >= sx && kxs < sx + kx) ? 0.f : -INFINITY;
  }

  // ---- per-tile y geometry: which stages each tile touches / needs a y mask in ----
  uint32_t act_mask[NTY], ym_mask[NTY];
  int syl[NTY], qyl[NTY];
#pragma unroll
  for (int tt = 0; tt < NTY; ++tt) {
    const int yt0 = y0 + tt * TY;
    if (yt0 < qy1) {
      const int ytl = min(yt0 + TY - 1, qy1 - 1);
      const int U0 = win_start(yt0, Ly, ky) - Y0, U1 = win_start(ytl, Ly, ky) + ky - Y0;  // union rows
      const int F0 = win_start(ytl, Ly, ky) - Y0, F1 = win_start(yt0, Ly, ky) + ky - Y0;  // rows in every window
      act_mask[tt] = bit_range(U0 / RPS, (U1 + RPS - 1) / RPS);
      ym_mask[tt] = act_mask[tt] & ~bit_range((F0 + RPS - 1) / RPS, F1 / RPS);
    } else {
      act_mask[tt] = ym_mask[tt] = 0;
    }
    qyl[tt] = yt0 + n16 / TX;
    syl[tt] = win_start(min(qyl[tt], qy1 - 1), Ly, ky) - Y0;
  }

  // ---- Q operands and each query's score against its own key ----
  const int rz = gz + dz * iz;
  const int rqx = gx + dx * qxc;
  const float c2 = p.scale * 1.4426950408889634f;  // scores in log2 units
  bf16x8 qreg[NTY][KS];
  float mref[NTY];
  {
    bf16x8 kself[NTY][KS];
#pragma unroll
    for (int tt = 0; tt < NTY; ++tt) {
      const int rqy = gy + dy * min(qyl[tt], qy1 - 1);
      const bf16* qp = (const bf16*)p.q + (int64_t)b * p.qs[0] + (int64_t)rz * p.qs[1] + (int64_t)rqy * p.qs[2] +
                       (int64_t)rqx * p.qs[3] + (int64_t)h * p.qs[4];
      const bf16* kp = (const bf16*)p.k + (int64_t)b * p.ks[0] + (int64_t)rz * p.ks[1] + (int64_t)rqy * p.ks[2] +
                       (int64_t)rqx * p.ks[3] + (int64_t)h * p.ks[4];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        qreg[tt][ks] = *(const bf16x8*)(qp + 32 * ks + 8 * g);
        kself[tt][ks] = *(const bf16x8*)(kp + 32 * ks + 8 * g);
      }
      if constexpr (ROPE && D == 64) {
        {  // the queries' rotation, pairs 8g .. 8g + 7 of this lane
          const int64_t ro = rope_row(p, b, rz, rqy, rqx) * 32 + 8 * g;
          float c[8], sn[8];
          *(f32x4*)&c[0] = *(const f32x4*)(p.rc + ro);
          *(f32x4*)&c[4] = *(const f32x4*)(p.rc + ro + 4);
          *(f32x4*)&sn[0] = *(const f32x4*)(p.rs + ro);
          *(f32x4*)&sn[4] = *(const f32x4*)(p.rs + ro + 4);
          rope_q_pairs(qreg[tt][0], qreg[tt][1], c, sn);
        }
      }
    }
    // Q must land before the DMA ring starts: the compiler does not see the
    // ring's loads, so a deferred wait for Q inside the loop would drain them.
    wait_vmcnt(0);
#pragma unroll
    for (int tt = 0; tt < NTY; ++tt) {
      float d = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          qreg[tt][ks][e] = (bf16)((float)qreg[tt][ks][e] * c2);  // scores in log2 units
          d = fmaf((float)qreg[tt][ks][e], (float)kself[tt][ks][e], d);
        }
      mref[tt] = colsum(d);
    }
  }

  // ---- DMA descriptors ----
  // A stage is 2*RPS regions (K rows 0..RPS-1, V rows 0..RPS-1), each LWP keys
  // of D bf16 in swizzled 16-byte chunks; wave w loads 1-KiB chunks w, w+4, ...
  // One buffer descriptor per tensor covers the stage's rows (the row offset is
  // part of the lane offset; the record count stops at the last valid row, so
  // rows past the window union read as zero).
  const int64_t rowk = 2 * (int64_t)dy * p.ks[2], rowv = 2 * (int64_t)dy * p.vs[2];  // bytes per sub-grid row
  uint32_t voff[LPT];
  bool vten[LPT];
#pragma unroll
  for (int j = 0; j < LPT; ++j) {
    const int gc = j * NWX + wave;  // 1-KiB chunk of the stage
    const int reg = gc / RKB;
    const int tensor = reg / RPS, row = reg % RPS;
    const int key = (gc % RKB) * KPK + lane / CPK;
    const int c = swz<D>(lane % CPK, key);  // logical chunk stored at this slot
    const int64_t sx3 = tensor ? p.vs[3] : p.ks[3];
    const int64_t rowb = tensor ? rowv : rowk;
    voff[j] = (key < LW && X0 + key < Lx)
                  ? (uint32_t)(row * rowb + (int64_t)(gx + dx * (X0 + key)) * sx3 * 2 + 16 * c)
                  : OOB;
    vten[j] = tensor;
  }
  // Issue cursor: row group `cp` (outer), z-slice `cz` (inner): the kz slices
  // of a row group are fetched back to back, so workgroups at neighbouring z
  // read the same rows close together in time (L2 reuse across the z window).
  const char* kp0 = (const char*)p.k + 2 * ((int64_t)b * p.ks[0] + (int64_t)h * p.ks[4] +
                                           (int64_t)(gz + dz * sz) * p.ks[1] + (int64_t)(gy + dy * Y0) * p.ks[2]);
  const char* vp0 = (const char*)p.v + 2 * ((int64_t)b * p.vs[0] + (int64_t)h * p.vs[4] +
                                           (int64_t)(gz + dz * sz) * p.vs[1] + (int64_t)(gy + dy * Y0) * p.vs[2]);
  const int64_t zstepk = 2 * (int64_t)dz * p.ks[1], zstepv = 2 * (int64_t)dz * p.vs[1];
  int cz = 0, cp = 0;
  const char* kcur = kp0;
  const char* vcur = vp0;
  uint32_t issue_off = 0;  // LDS byte offset of the ring slot the cursor fills

  auto issue = [&]() {
    const int nrow = min(max(NR - RPS * cp, 0), RPS);  // valid rows of the stage at the cursor
    const uint32_t nk = (uint32_t)(nrow * rowk);
    const uint32_t nv = (uint32_t)(nrow * rowv);
    const u32x4 rk = make_rsrc(kcur, nk);
    const u32x4 rv = make_rsrc(vcur, nv);
    const uint32_t m0 = lds_base + issue_off + (uint32_t)wave * 1024;
#pragma unroll
    for (int j = 0; j < LPT; ++j) dma_row16(vten[j] ? rv : rk, m0 + j * NWX * 1024, voff[j]);
    // advance the cursor
    issue_off = issue_off + STAGE_B == NBUF * STAGE_B ? 0 : issue_off + STAGE_B;
    if (++cz == kz) {
      cz = 0;
      ++cp;
      kp0 += RPS * rowk;
      vp0 += RPS * rowv;
      kcur = kp0;
      vcur = vp0;
    } else {
      kcur += zstepk;
      vcur += zstepv;
    }
  };

  // ---- LDS read offsets (bytes within a stage) ----
  uint32_t koff[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int key = off_w + n16;
    koff[ks] = (key * D + 8 * swz<D>(4 * ks + g, key)) * 2;
  }
  uint32_t voffs[DB];
  {
    const int keyv = off_w + 4 * g + (n16 >> 2);
    const int dq = n16 & 3;
#pragma unroll
    for (int db = 0; db < DB; ++db)
      voffs[db] = RPS * RB + (keyv * D + 8 * swz<D>(2 * db + (dq >> 1), keyv) + 4 * (dq & 1)) * 2;
  }

  f32x4 oacc[NTY][DB];
  f32x4 lacc[NTY];
  f32x4 nb[NTY];  // xbias - mref: the C operand of the QK MFMA
#pragma unroll
  for (int tt = 0; tt < NTY; ++tt) {
#pragma unroll
    for (int db = 0; db < DB; ++db) oacc[tt][db] = (f32x4){0.f, 0.f, 0.f, 0.f};
    lacc[tt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i) nb[tt][i] = xbias[i] - mref[tt];
  }
  typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
  bf16x8_t ones = {(bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f};

#pragma unroll
  for (int s = 0; s < NBUF - 1; ++s) issue();

  uint32_t cur_off = 0;  // ring slot of the stage being computed
  int pr = 0, zc = 0;
  for (int s = 0; s < nstage; ++s) {
    wait_vmcnt((NBUF - 2) * LPT);  // constant: the tail issues empty (zero-record) stages
    lds_barrier();
    issue();

    asm volatile("" : "+v"(ones));  // keep the ones operand resident (else rebuilt per tile)
    const char* st = lds + cur_off;
    bf16x8 ak[RPS][KS];
#pragma unroll
    for (int r = 0; r < RPS; ++r)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) ak[r][ks] = *(const bf16x8*)(st + r * RB + koff[ks]);
    bf16x8 av[NRP][DB];  // V^T of row pair rp: keys of row 2rp then row 2rp+1
#pragma unroll
    for (int rp = 0; rp < NRP; ++rp)
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_PTR(bf16x4, st + voffs[db] + 2 * rp * RB));
        const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_PTR(bf16x4, st + voffs[db] + (2 * rp + 1) * RB));
        av[rp][db] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      }
    const int r0 = RPS * pr;

#pragma unroll
    for (int tt = 0; tt < NTY; ++tt) {
      if (!((act_mask[tt] >> pr) & 1)) continue;  // rows outside this tile's window union
      f32x4 sacc[RPS];
#pragma unroll
      for (int r = 0; r < RPS; ++r) {
        sacc[r] = nb[tt];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          sacc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ak[r][ks], qreg[tt][ks], sacc[r], 0, 0, 0);
      }
      float u[4 * RPS];
#pragma unroll
      for (int r = 0; r < RPS; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) u[4 * r + i] = sacc[r][i];
      if ((ym_mask[tt] >> pr) & 1) {
        // a row outside some query's y window (else only the x mask applies)
#pragma unroll
        for (int r = 0; r < RPS; ++r) {
          const int yr = r0 + r;
          const bool yok = yr >= syl[tt] && yr < syl[tt] + ky;
#pragma unroll
          for (int i = 0; i < 4; ++i) u[4 * r + i] = yok ? u[4 * r + i] : -INFINITY;
        }
      }
      // The reference only has to move when some score exceeds it by TAU; the
      // in-lane max decides that, the column max is needed only to move it.
      float ml = -INFINITY;
#pragma unroll
      for (int j = 0; j < 4 * RPS; j += 8)
        ml = fmaxf(ml, fmaxf(fmaxf(fmaxf(u[j], u[j + 1]), u[j + 2]),
                             fmaxf(fmaxf(fmaxf(u[j + 3], u[j + 4]), u[j + 5]), fmaxf(u[j + 6], u[j + 7]))));
      if (__builtin_amdgcn_ballot_w64(ml > TAU) != 0) {
        const float mx = colmax(ml);
        const float d = mx > TAU ? mx : 0.f;
        const float alpha = __builtin_amdgcn_exp2f(-d);
#pragma unroll
        for (int db = 0; db < DB; ++db) oacc[tt][db] *= alpha;
        lacc[tt] *= alpha;
        mref[tt] += d;
#pragma unroll
        for (int i = 0; i < 4; ++i) nb[tt][i] -= d;
#pragma unroll
        for (int j = 0; j < 4 * RPS; ++j) u[j] -= d;
      }
      // One straight-line block: P of every row pair, then the PV MFMAs.
      bf16x8 pb[NRP];
#pragma unroll
      for (int rp = 0; rp < NRP; ++rp) {
        float pv[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) pv[j] = __builtin_amdgcn_exp2f(u[8 * rp + j]);
        const u32x4 pw = {pack_bf16x2(pv[0], pv[1]), pack_bf16x2(pv[2], pv[3]), pack_bf16x2(pv[4], pv[5]),
                          pack_bf16x2(pv[6], pv[7])};
        pb[rp] = __builtin_bit_cast(bf16x8, pw);
      }
#pragma unroll
      for (int rp = 0; rp < NRP; ++rp) {
        lacc[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pb[rp], lacc[tt], 0, 0, 0);
#pragma unroll
        for (int db = 0; db < DB; ++db)
          oacc[tt][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[rp][db], pb[rp], oacc[tt][db], 0, 0, 0);
      }
    }
    cur_off = cur_off + STAGE_B == NBUF * STAGE_B ? 0 : cur_off + STAGE_B;
    if (++zc == kz) {  // stages run row-group-major, z-minor
      zc = 0;
      ++pr;
    }
  }
  wait_vmcnt(0);

  // ---- normalise and store ----
#pragma unroll
  for (int tt = 0; tt < NTY; ++tt) {
    const int qy = qyl[tt];
    if (qy >= qy1 || qx >= qx1) continue;
    const float inv = 1.f / lacc[tt][0];
    const int oz = rz - p.org[0];
    const int oy = gy + dy * qy - p.org[1];
    const int ox = gx + dx * qx - p.org[2];
    if (p.lse && g == 0) p.lse[lse_index(p, b, oz, oy, ox, h)] = mref[tt] + __log2f(lacc[tt][0]);
    bf16* op = (bf16*)p.o + (int64_t)b * p.os[0] + (int64_t)oz * p.os[1] + (int64_t)oy * p.os[2] +
               (int64_t)ox * p.os[3] + (int64_t)h * p.os[4];
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const u32x2 w = {pack_bf16x2(oacc[tt][db][0] * inv, oacc[tt][db][1] * inv),
                       pack_bf16x2(oacc[tt][db][2] * inv, oacc[tt][db][3] * inv)};
      *(u32x2*)(op + 16 * db + 4 * g) = w;
    }
  }
#endif
}

// Two workgroups per CU for head_dim <= 64; head_dim 128 needs the full register file.
template <int D, int TX, int NTY, int RPS, int NBUF>
__global__ __launch_bounds__(256, 2) void na3d_mfma_kernel(Na3dParams p, Na3dTiles tg) {
  __shared__ __attribute__((aligned(1024))) char lds[mfma_lds_bytes<D, TX, RPS, NBUF>()];
  na3d_mfma_body<D, TX, NTY, RPS, NBUF>(p, tg, lds, (int)__builtin_amdgcn_workgroup_id_x());
}
template <int D, int TX, int NTY, int RPS, int NBUF>
__global__ __launch_bounds__(256, 1) void na3d_mfma_wide_kernel(Na3dParams p, Na3dTiles tg) {
  __shared__ __attribute__((aligned(1024))) char lds[mfma_lds_bytes<D, TX, RPS, NBUF>()];
  na3d_mfma_body<D, TX, NTY, RPS, NBUF>(p, tg, lds, (int)__builtin_amdgcn_workgroup_id_x());
}

// ---------------------------------------------------------------------------
// Strip kernel: one workgroup walks a whole column of query tiles along y
// ---------------------------------------------------------------------------
// Work unit: (batch, head, dilation residue, z, 4*TX query columns) and a
// chunk of query rows [ys, ye) (the whole y range unless that leaves too few
// workgroups).  The chunk's tiles of (TY, TX) queries are j = 0, 1, ... along
// y; tile j needs the key rows U_j = [ws(first row), ws(last row) + ky) of
// every z-slice of the window.  Key rows stream through the LDS ring once, in
// groups of RPS rows (all kz slices of a group back to back), and each group
// feeds every tile whose union it meets.  A wave keeps four tiles in flight in
// four register slots (tile j in slot j & 3): when a tile's union has passed
// it is normalised and stored, and the tile four rows further takes its slot.
// For an unclamped window with ky + TY - 1 = 4 * RPS (configs like 3x13x13
// with 4x4 tiles) every group feeds exactly four tiles with all its rows,
// where a fixed box of four tiles per wave is active in only ky+3 of
// ky+15 rows.
//
// Clamped windows at the grid's edges can make tile j + 4 start before tile
// j has finished, or two tiles start in one group.  The walk is then split
// into segments: a new segment starts at such a tile and streams from its
// union's first row again (a few groups are read twice; exact results).
//
// Q and the query's own key (which seeds the softmax reference) of the tile
// that starts in group g + 1 are copied into LDS while group g runs; the
// tiles that start in a segment's first group are staged through the ring.
struct Na3dStrips {
  int nxt, nzt;  // query column boxes and z-slices per (batch, head, residue)
  int nch, cty;  // y chunks and tiles per chunk
  int nres;      // dil_z * dil_y * dil_x
  int total;     // workgroups in the launch
};


// Where one strip tile's queries sit: batch, head, residue (gz, gy, gx), the
// tile's sub-grid z, first query row and first column, and the chunk's ends.
struct StripTile {
  int b, h, gz, gy, gx, iz, qy0, ye, qx0, qx1;
};

// Rare path of the strip kernels: recompute one (16/TX) x TX tile of queries
// exactly, straight from global memory, with a running maximum (fp32 online
// softmax).  Called by a whole wave when the tile's unnormalised sums left the
// range the fast path guarantees (scores far from 0 in log2 units, or
// non-finite inputs).  Lane l handles query l >> 2 (row-major in the tile)
// and the head-dim quarter l & 3 (16 values); invalid queries (past the
// chunk's last row or column) compute a clamped copy and store nothing.
template <int TX = 4, bool ROPE = false>
__device__ __forceinline__ void na3d_strip_tile_exact(const Na3dParams* pp, StripTile t) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int TY = 16 / TX;
  const Na3dParams& p = *pp;
  const int lane = (int)__builtin_amdgcn_workitem_id_x() & 63;
  const int n = lane >> 2, dq = lane & 3;
  const int dz = p.dil[0], dy = p.dil[1], dx = p.dil[2];
  const int Lz = sub_len(p.L[0], t.gz, dz), Ly = sub_len(p.L[1], t.gy, dy), Lx = sub_len(p.L[2], t.gx, dx);
  static_assert(TX * TY == 16, "16 queries per tile");
  const bool valid = t.qy0 + n / TX < t.ye && t.qx0 + n % TX < t.qx1;
  const int qy = min(t.qy0 + n / TX, t.ye - 1), qx = min(t.qx0 + n % TX, t.qx1 - 1);
  const int sz = win_start(t.iz, Lz, p.ker[0]), sy = win_start(qy, Ly, p.ker[1]), sx = win_start(qx, Lx, p.ker[2]);
  const int rz = t.gz + dz * t.iz, ry = t.gy + dy * qy, rx = t.gx + dx * qx;
  const bf16* qp = (const bf16*)p.q + (int64_t)t.b * p.qs[0] + (int64_t)rz * p.qs[1] + (int64_t)ry * p.qs[2] +
                   (int64_t)rx * p.qs[3] + (int64_t)t.h * p.qs[4] + 16 * dq;
  const float c2 = p.scale * 1.4426950408889634f;
  float qf[16], acc[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    qf[i] = (float)qp[i];
    acc[i] = 0.f;
  }
  if constexpr (ROPE) {  // the queries' rotation (head_dim 64): this lane's dims 16dq .. 16dq + 15, partners 32 apart
    const bf16* pp2 = dq < 2 ? qp + 32 : qp - 32;
    const int64_t ro = rope_row(p, t.b, rz, ry, rx) * 32 + 16 * (dq & 1);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float o = qf[i], q2 = (float)pp2[i], c = p.rc[ro + i], sn = p.rs[ro + i];
      // dims d < 32: a = own, b = partner (a c - b s); d >= 32: a = partner, b = own (a s + b c)
      qf[i] = (float)(bf16)(dq < 2 ? rope_rot_a(o, q2, c, sn) : rope_rot_b(q2, o, c, sn));
    }
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) qf[i] *= c2;
  float m = -INFINITY, l = 0.f;
  const bf16* kb = (const bf16*)p.k + (int64_t)t.b * p.ks[0] + (int64_t)t.h * p.ks[4] + 16 * dq;
  const bf16* vb = (const bf16*)p.v + (int64_t)t.b * p.vs[0] + (int64_t)t.h * p.vs[4] + 16 * dq;
  for (int a = 0; a < p.ker[0]; ++a) {
    const int kzr = t.gz + dz * (sz + a);
    for (int c = 0; c < p.ker[1]; ++c) {
      const int kyr = t.gy + dy * (sy + c);
      for (int e = 0; e < p.ker[2]; ++e) {
        const int kxr = t.gx + dx * (sx + e);
        const bf16* kp = kb + (int64_t)kzr * p.ks[1] + (int64_t)kyr * p.ks[2] + (int64_t)kxr * p.ks[3];
        const bf16* vp = vb + (int64_t)kzr * p.vs[1] + (int64_t)kyr * p.vs[2] + (int64_t)kxr * p.vs[3];
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) s = fmaf(qf[i], (float)kp[i], s);
        s += __shfl_xor(s, 1);
        s += __shfl_xor(s, 2);
        const float mn = fmaxf(m, s);
        const float alpha = exp2f(m - mn), w = exp2f(s - mn);
        l = l * alpha + w;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = fmaf(acc[i], alpha, w * (float)vp[i]);
        m = mn;
      }
    }
  }
  if (!valid) return;
  if (p.lse && dq == 0) p.lse[lse_index(p, t.b, rz - p.org[0], ry - p.org[1], rx - p.org[2], t.h)] = m + __log2f(l);
  const float inv = 1.f / l;
  char* op = (char*)p.o + 2 * ((int64_t)t.b * p.os[0] + (int64_t)(rz - p.org[0]) * p.os[1] +
                               (int64_t)(ry - p.org[1]) * p.os[2] + (int64_t)(rx - p.org[2]) * p.os[3] +
                               (int64_t)t.h * p.os[4] + 16 * dq);
#pragma unroll
  for (int i = 0; i < 16; i += 8) {
    const u32x4 w = {pack_bf16x2(acc[i] * inv, acc[i + 1] * inv), pack_bf16x2(acc[i + 2] * inv, acc[i + 3] * inv),
                     pack_bf16x2(acc[i + 4] * inv, acc[i + 5] * inv), pack_bf16x2(acc[i + 6] * inv, acc[i + 7] * inv)};
    *(u32x4*)(op + 2 * i) = w;
  }
#endif
}

template <int D, int TX, int RPS, int NBUF>
__device__ __forceinline__ void na3d_strip_body(const Na3dParams p, const Na3dStrips sg) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int NWX = NA3D_NWX;
  constexpr int NS = 4;                   // tile slots per wave
  constexpr int TY = 16 / TX;
  constexpr int WQX = NWX * TX;           // workgroup query columns
  constexpr int LW = (NWX - 1) * TX + 16; // keys per LDS row that are read
  constexpr int KPK = 512 / D;            // keys per KiB
  constexpr int LWP = (LW + KPK - 1) / KPK * KPK;
  constexpr int RB = LWP * D * 2;         // bytes per (tensor, row) region
  constexpr int RKB = RB / 1024;
  constexpr int STAGE_B = 2 * RPS * RB;   // K rows 0..RPS-1, then V rows 0..RPS-1
  constexpr int LPT = 2 * RPS * RKB / NWX;  // 1-KiB DMA loads per wave per stage
  constexpr int NRP = RPS / 2;
  constexpr int CPK = D / 8;              // 16-byte chunks per key
  constexpr int KS = D / 32;              // k-steps of the QK MFMA; also 1-KiB loads per wave for 16 query rows
  constexpr int DB = D / 16;
  constexpr int QWB = 16 * D * 2;         // one wave's 16 rows of Q (or of self keys), bytes
  constexpr int QTB = NWX * 2 * QWB;      // Q and self keys of one tile row of the workgroup
  constexpr int RING_B = NBUF * STAGE_B;
  constexpr float TAU = 64.f;             // lazy-rescale slack, log2 units (as in na3d_mfma_body)
  static_assert(RKB == NWX && (RPS == 2 || RPS == 4), "stage layout: wave w loads the w-th KiB of every row");
  static_assert(LPT == 2 * RPS, "a wave loads the same key block of every row of a stage");
  static_assert(QWB == KS * 1024, "16 query rows are KS 1-KiB loads");
  static_assert(NS * QTB <= RING_B, "a segment's first tiles are staged through the ring");
  static_assert(TY <= RPS, "at most one tile starts per group");

  __shared__ __attribute__((aligned(1024))) char lds[RING_B + QTB];

  // ---- work unit ----
  int t = xcd_tile_order(sg.total, (int)__builtin_amdgcn_workgroup_id_x());
  const int xb = t % sg.nxt;
  t /= sg.nxt;
  const int zt = t % sg.nzt;
  t /= sg.nzt;
  const int ch = t % sg.nch;
  t /= sg.nch;
  const int res = t % sg.nres;
  t /= sg.nres;
  const int h = t % p.H;
  const int b = t / p.H;
  const int dz = p.dil[0], dy = p.dil[1], dx = p.dil[2];
  const int gx = res % dx;
  const int gy = (res / dx) % dy;
  const int gz = res / (dx * dy);

  const int Lz = sub_len(p.L[0], gz, dz);
  const int Ly = sub_len(p.L[1], gy, dy);
  const int Lx = sub_len(p.L[2], gx, dx);
  const int qz0 = sub_first(p.org[0], gz, dz), qz1 = sub_end(p.org[0], p.ext[0], gz, dz);
  const int qy0 = sub_first(p.org[1], gy, dy), qy1 = sub_end(p.org[1], p.ext[1], gy, dy);
  const int qx0 = sub_first(p.org[2], gx, dx), qx1 = sub_end(p.org[2], p.ext[2], gx, dx);
  const int iz = qz0 + zt;
  const int ys = qy0 + ch * sg.cty * TY;
  const int ye = min(ys + sg.cty * TY, qy1);
  const int x0 = qx0 + xb * WQX;
  if (iz >= qz1 || ys >= ye || x0 >= qx1) return;  // uniform over the workgroup
  const int NT = (ye - ys + TY - 1) / TY;

  const int kz = p.ker[0], ky = p.ker[1], kx = p.ker[2];
  const int sz = win_start(iz, Lz, kz);
  const int X0 = win_start(x0, Lx, kx);

  const int tid = (int)__builtin_amdgcn_workitem_id_x();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int n16 = lane & 15;
  const int g = lane >> 4;
  const int trow = n16 / TX;  // this lane's query row within a tile
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;

  // ---- per-lane x geometry (shared by every tile of the wave) ----
  const int xw0 = x0 + wave * TX;
  const int off_w = win_start(min(xw0, qx1 - 1), Lx, kx) - X0;
  const int qx = xw0 + n16 % TX;
  uint32_t xmask = 0;  // bit i: key 4g+i of the wave's block is outside this lane's x window
  {
    const int sx = win_start(min(qx, qx1 - 1), Lx, kx);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int kxs = X0 + off_w + 4 * g + i;
      xmask |= (kxs >= sx && kxs < sx + kx) ? 0u : (1u << i);
    }
  }

  // Union [u0, u1) of tile j's windows and the rows [f0, f1) inside all of them.
  auto tile_rows = [&](int j, int& u0, int& u1, int& f0, int& f1) {
    const int y = ys + TY * j;
    const int yl = min(y + TY - 1, ye - 1);
    const int w0 = win_start(y, Ly, ky), w1 = win_start(yl, Ly, ky);
    u0 = w0;
    u1 = w1 + ky;
    f0 = w1;
    f1 = w0 + ky;
  };

  const int rz = gz + dz * iz;
  const float c2 = p.scale * 1.4426950408889634f;  // scores in log2 units

  // ---- K/V ring lane offsets: wave w loads keys [w*KPK, (w+1)*KPK) of every row ----
  const int64_t rowk = 2 * (int64_t)dy * p.ks[2], rowv = 2 * (int64_t)dy * p.vs[2];
  uint32_t xoffk, xoffv;
  {
    const int key = (wave % RKB) * KPK + lane / CPK;
    const int c = swz<D>(lane % CPK, key);
    const bool in = key < LW && X0 + key < Lx;
    xoffk = in ? (uint32_t)((int64_t)(gx + dx * (X0 + key)) * p.ks[3] * 2 + 16 * c) : OOB;
    xoffv = in ? (uint32_t)((int64_t)(gx + dx * (X0 + key)) * p.vs[3] * 2 + 16 * c) : OOB;
  }
  // ---- Q and self-key copies: one (batch, z, head) slice, 31-bit offsets ----
  const u32x4 rq = make_rsrc((const char*)p.q + 2 * ((int64_t)b * p.qs[0] + (int64_t)rz * p.qs[1] + (int64_t)h * p.qs[4]),
                             0x7fffffffu);
  const u32x4 rks = make_rsrc((const char*)p.k + 2 * ((int64_t)b * p.ks[0] + (int64_t)rz * p.ks[1] + (int64_t)h * p.ks[4]),
                              0x7fffffffu);
  const uint32_t qs2 = (uint32_t)(2 * dy * p.qs[2]), ks2 = (uint32_t)(2 * dy * p.ks[2]);
  uint32_t qxo[KS], kxo[KS];  // x part of the lane's offsets; y part added per tile
#pragma unroll
  for (int i = 0; i < KS; ++i) {
    const int n = lane / CPK + i * (64 / CPK);
    const int rx = gx + dx * min(xw0 + n % TX, qx1 - 1);
    qxo[i] = (uint32_t)((int64_t)rx * p.qs[3] * 2 + (int64_t)gy * p.qs[2] * 2) + 16 * (lane % CPK);
    kxo[i] = (uint32_t)((int64_t)rx * p.ks[3] * 2 + (int64_t)gy * p.ks[2] * 2) + 16 * (lane % CPK);
  }
  // Copy Q and the self keys of tile j (this wave's 16 queries) to LDS at `off`:
  // query n's row at n*2D bytes, self keys QWB further.
  auto dma_q = [&](int j, uint32_t off) {
    const int yt0 = ys + TY * j;
    const uint32_t m0 = lds_base + off + (uint32_t)wave * 2 * QWB;
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      const int n = lane / CPK + i * (64 / CPK);
      const uint32_t qy = (uint32_t)min(yt0 + n / TX, ye - 1);
      dma_row16(rq, m0 + i * 1024, qxo[i] + qy * qs2);
      dma_row16(rks, m0 + QWB + i * 1024, kxo[i] + qy * ks2);
    }
  };
  // ---- output: one (batch, z, head) slice, lane offset of its column and row 0 ----
  char* obase = (char*)p.o + 2 * ((int64_t)b * p.os[0] + (int64_t)(rz - p.org[0]) * p.os[1] + (int64_t)h * p.os[4]);
  const int64_t orow = 2 * (int64_t)dy * p.os[2];
  const int64_t ooff = 2 * ((int64_t)(gx + dx * qx - p.org[2]) * p.os[3] + (int64_t)(gy - p.org[1]) * p.os[2]) + 8 * g;

  // ---- LDS read offsets of the K/V operands (bytes within a stage) ----
  uint32_t koff[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int key = off_w + n16;
    koff[ks] = (key * D + 8 * swz<D>(4 * ks + g, key)) * 2;
  }
  uint32_t voffs[DB];
  {
    const int keyv = off_w + 4 * g + (n16 >> 2);
    const int dq = n16 & 3;
#pragma unroll
    for (int db = 0; db < DB; ++db)
      voffs[db] = RPS * RB + (keyv * D + 8 * swz<D>(2 * db + (dq >> 1), keyv) + 4 * (dq & 1)) * 2;
  }

  // ---- tile slots ----
  bf16x8 qreg[NS][KS];
  f32x4 oacc[NS][DB];
  f32x4 lacc[NS];
  f32x4 nb[NS];  // x bias - reference: the C operand of the QK MFMA
  int syl[NS];   // first window row of this lane's query row (relative to the segment)
  float mslot[NS];  // the slot's softmax reference (log2 units), for the lse output
  // Uniform slot state: tile index (-1: empty) and packed groups
  // [ylo | yhi << 10 | end << 20]: groups below ylo or from yhi on have rows
  // outside some query's window; `end` is the tile's last group.
  int s_tile[NS], s_grp[NS];
#pragma unroll
  for (int k = 0; k < NS; ++k) s_tile[k] = -1, s_grp[k] = 0;
  typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
  bf16x8_t ones = {(bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f};

  int S = 0;  // first key row of the current segment
  // Tile j enters slot k: Q (pre-scaled) and its score against its own key from LDS.
  auto start_tile = [&](int k, int j, uint32_t off) {
    const char* qb = lds + off + wave * 2 * QWB;
    bf16x8 kself[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      qreg[k][ks] = *(const bf16x8*)(qb + n16 * D * 2 + (4 * ks + g) * 16);
      kself[ks] = *(const bf16x8*)(qb + QWB + n16 * D * 2 + (4 * ks + g) * 16);
    }
    float d = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        qreg[k][ks][e] = (bf16)((float)qreg[k][ks][e] * c2);
        d = fmaf((float)qreg[k][ks][e], (float)kself[ks][e], d);
      }
    const float mref = colsum(d);
    mslot[k] = mref;
#pragma unroll
    for (int i = 0; i < 4; ++i) nb[k][i] = ((xmask >> i) & 1) ? -INFINITY : -mref;
#pragma unroll
    for (int db = 0; db < DB; ++db) oacc[k][db] = (f32x4){0.f, 0.f, 0.f, 0.f};
    lacc[k] = (f32x4){0.f, 0.f, 0.f, 0.f};
    int u0, u1, f0, f1;
    tile_rows(j, u0, u1, f0, f1);
    s_tile[k] = j;
    s_grp[k] = (f0 - S + RPS - 1) / RPS | ((f1 - S) / RPS) << 10 | ((u1 - 1 - S) / RPS) << 20;
    syl[k] = win_start(min(ys + TY * j + trow, ye - 1), Ly, ky) - S;
  };
  auto finish_tile = [&](int k) {
    const int qy = ys + TY * s_tile[k] + trow;
    s_tile[k] = -1;
    if (qy >= ye || qx >= qx1) return;
    const float inv = 1.f / lacc[k][0];
    if (p.lse && g == 0)
      p.lse[lse_index(p, b, rz - p.org[0], gy + dy * qy - p.org[1], gx + dx * qx - p.org[2], h)] =
          mslot[k] + __log2f(lacc[k][0]);
    char* op = obase + ooff + (int64_t)qy * orow;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const u32x2 w = {pack_bf16x2(oacc[k][db][0] * inv, oacc[k][db][1] * inv),
                       pack_bf16x2(oacc[k][db][2] * inv, oacc[k][db][3] * inv)};
      *(u32x2*)(op + 32 * db) = w;
    }
  };

  const int64_t zstepk = 2 * (int64_t)dz * p.ks[1], zstepv = 2 * (int64_t)dz * p.vs[1];
  const char* kz0 = (const char*)p.k + 2 * ((int64_t)b * p.ks[0] + (int64_t)h * p.ks[4] + (int64_t)(gz + dz * sz) * p.ks[1] +
                                           (int64_t)gy * p.ks[2]);
  const char* vz0 = (const char*)p.v + 2 * ((int64_t)b * p.vs[0] + (int64_t)h * p.vs[4] + (int64_t)(gz + dz * sz) * p.vs[1] +
                                           (int64_t)gy * p.vs[2]);
  int js = 0;
  while (js < NT) {
    // ---- segment [js, je]: no slot conflict, at most one start per later group ----
    int u0, u1, f0, f1;
    tile_rows(js, u0, u1, f0, f1);
    S = u0;
    int je = js, prev_a = 0;
    while (je + 1 < NT) {
      const int j = je + 1;
      tile_rows(j, u0, u1, f0, f1);
      const int aj = (u0 - S) / RPS;
      if (aj > 0 && aj == prev_a) break;
      if (j - NS >= js) {
        int v0, v1, e0, e1;
        tile_rows(j - NS, v0, v1, e0, e1);
        if (aj <= (v1 - 1 - S) / RPS) break;
      }
      prev_a = aj;
      je = j;
    }
    tile_rows(je, u0, u1, f0, f1);
    const int NR = u1 - S;  // key rows the segment streams
    const int nstage = kz * ((NR + RPS - 1) / RPS);

    // ---- tiles that start in the first group: Q staged through the ring ----
    lds_barrier();  // the previous segment's ring reads are done
    int jn = js;
    for (; jn <= je; ++jn) {
      tile_rows(jn, u0, u1, f0, f1);
      if (u0 - S >= RPS) break;
      dma_q(jn, (uint32_t)((jn - js) * QTB));
    }
    wait_vmcnt(0);
#pragma unroll
    for (int k = 0; k < NS; ++k)
      for (int j = js; j < jn; ++j)
        if ((j & (NS - 1)) == k) start_tile(k, j, (uint32_t)((j - js) * QTB));
    wait_lgkm0();
    lds_barrier();  // staged Q read before the ring overwrites it
    int a_next = NR;  // first group of tile jn
    if (jn <= je) {
      tile_rows(jn, u0, u1, f0, f1);
      a_next = (u0 - S) / RPS;
    }

    // ---- K/V ring over the segment's rows, row-group-major, z-minor ----
    const char* kseg = kz0 + (int64_t)S * rowk;
    const char* vseg = vz0 + (int64_t)S * rowv;
    int cz = 0, cp = 0;
    uint32_t issue_off = 0;
    auto issue = [&]() {
      const int nrow = min(max(NR - RPS * cp, 0), RPS);
      const u32x4 rk = make_rsrc(kseg + (int64_t)cp * RPS * rowk + (int64_t)cz * zstepk, (uint32_t)(nrow * rowk));
      const u32x4 rv = make_rsrc(vseg + (int64_t)cp * RPS * rowv + (int64_t)cz * zstepv, (uint32_t)(nrow * rowv));
      const uint32_t m0 = lds_base + issue_off + (uint32_t)(wave / RKB) * RB + (uint32_t)(wave % RKB) * 1024;
#pragma unroll
      for (int r = 0; r < RPS; ++r) dma_row16(rk, m0 + r * RB, xoffk + (uint32_t)(r * rowk));
#pragma unroll
      for (int r = 0; r < RPS; ++r) dma_row16(rv, m0 + (RPS + r) * RB, xoffv + (uint32_t)(r * rowv));
      issue_off = issue_off + STAGE_B == RING_B ? 0 : issue_off + STAGE_B;
      if (++cz == kz) {
        cz = 0;
        ++cp;
      }
    };
#pragma unroll
    for (int s = 0; s < NBUF - 1; ++s) issue();

    uint32_t cur_off = 0;
    int gr = 0, zc = 0;  // group and z-slice of the stage being computed
    for (int s = 0; s < nstage; ++s) {
      const bool starting = zc == 0 && gr > 0 && gr == a_next;
      if (starting)
        wait_vmcnt(0);  // the tile's Q copy as well
      else
        wait_vmcnt((NBUF - 2) * LPT);
      lds_barrier();
      issue();
      if (starting) {
#pragma unroll
        for (int k = 0; k < NS; ++k)
          if ((jn & (NS - 1)) == k) start_tile(k, jn, (uint32_t)RING_B);
        ++jn;
        a_next = NR;
        if (jn <= je) {
          tile_rows(jn, u0, u1, f0, f1);
          a_next = (u0 - S) / RPS;
        }
      }
      // Q of the tile starting in the next group (each wave reads and refills
      // only its own part of the buffer; the start above has consumed it).
      if (zc == 1 && a_next == gr + 1) dma_q(jn, (uint32_t)RING_B);

      asm volatile("" : "+v"(ones));
      const char* st = lds + cur_off;
      bf16x8 ak[RPS][KS];
#pragma unroll
      for (int r = 0; r < RPS; ++r)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) ak[r][ks] = *(const bf16x8*)(st + r * RB + koff[ks]);
      bf16x8 av[NRP][DB];
#pragma unroll
      for (int rp = 0; rp < NRP; ++rp)
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_PTR(bf16x4, st + voffs[db] + 2 * rp * RB));
          const bf16x4 hi =
              __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_PTR(bf16x4, st + voffs[db] + (2 * rp + 1) * RB));
          av[rp][db] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
      const int r0 = RPS * gr;

#pragma unroll
      for (int k = 0; k < NS; ++k) {
        if (s_tile[k] < 0) continue;
        f32x4 sacc[RPS];
#pragma unroll
        for (int r = 0; r < RPS; ++r) {
          sacc[r] = nb[k];
#pragma unroll
          for (int ks = 0; ks < KS; ++ks)
            sacc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ak[r][ks], qreg[k][ks], sacc[r], 0, 0, 0);
        }
        float u[4 * RPS];
#pragma unroll
        for (int r = 0; r < RPS; ++r)
#pragma unroll
          for (int i = 0; i < 4; ++i) u[4 * r + i] = sacc[r][i];
        if (gr < (s_grp[k] & 1023) || gr >= ((s_grp[k] >> 10) & 1023)) {
          // rows outside some query's y window (else only the x mask applies)
#pragma unroll
          for (int r = 0; r < RPS; ++r) {
            const int yr = r0 + r;
            const bool yok = yr >= syl[k] && yr < syl[k] + ky;
#pragma unroll
            for (int i = 0; i < 4; ++i) u[4 * r + i] = yok ? u[4 * r + i] : -INFINITY;
          }
        }
        float ml = -INFINITY;
#pragma unroll
        for (int j = 0; j < 4 * RPS; j += 8)
          ml = fmaxf(ml, fmaxf(fmaxf(fmaxf(u[j], u[j + 1]), u[j + 2]),
                               fmaxf(fmaxf(fmaxf(u[j + 3], u[j + 4]), u[j + 5]), fmaxf(u[j + 6], u[j + 7]))));
        if (__builtin_amdgcn_ballot_w64(ml > TAU) != 0) {
          const float mx = colmax(ml);
          const float d = mx > TAU ? mx : 0.f;
          const float alpha = __builtin_amdgcn_exp2f(-d);
#pragma unroll
          for (int db = 0; db < DB; ++db) oacc[k][db] *= alpha;
          lacc[k] *= alpha;
          mslot[k] += d;
#pragma unroll
          for (int i = 0; i < 4; ++i) nb[k][i] -= d;
#pragma unroll
          for (int j = 0; j < 4 * RPS; ++j) u[j] -= d;
        }
        bf16x8 pb[NRP];
#pragma unroll
        for (int rp = 0; rp < NRP; ++rp) {
          float pv[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) pv[j] = __builtin_amdgcn_exp2f(u[8 * rp + j]);
          const u32x4 pw = {pack_bf16x2(pv[0], pv[1]), pack_bf16x2(pv[2], pv[3]), pack_bf16x2(pv[4], pv[5]),
                            pack_bf16x2(pv[6], pv[7])};
          pb[rp] = __builtin_bit_cast(bf16x8, pw);
        }
#pragma unroll
        for (int rp = 0; rp < NRP; ++rp) {
          lacc[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pb[rp], lacc[k], 0, 0, 0);
#pragma unroll
          for (int db = 0; db < DB; ++db)
            oacc[k][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[rp][db], pb[rp], oacc[k][db], 0, 0, 0);
        }
      }
      cur_off = cur_off + STAGE_B == RING_B ? 0 : cur_off + STAGE_B;
      if (++zc == kz) {
        zc = 0;
#pragma unroll
        for (int k = 0; k < NS; ++k)
          if (s_tile[k] >= 0 && (s_grp[k] >> 20) == gr) finish_tile(k);
        ++gr;
      }
    }
    wait_vmcnt(0);  // the ring's trailing (empty) stages
    js = je + 1;
  }
#endif
}

template <int D, int TX, int RPS, int NBUF>
__global__ __launch_bounds__(256, 2) void na3d_strip_kernel(Na3dParams p, Na3dStrips sg) {
  na3d_strip_body<D, TX, RPS, NBUF>(p, sg);
}


// ---------------------------------------------------------------------------
// Strip kernel, reference-free instance for regular strips
// ---------------------------------------------------------------------------
// Regular strip: ky = 13, 4x4 tiles, four key rows per group, and no query row
// of the chunk with a clamped y window (the host checks; configs like
// 3x13x13 on a halo-padded tile).  Then tile j's y-union is rows
// [4j, 4j + 16) of the strip: it starts in group j and ends in group j + 3,
// in slot j & 3, so in group gr the tile in its first group sits in slot
// gr & 3 and the one in its last group in slot (gr + 1) & 3.  The group loop
// is unrolled four times, which makes both slots compile-time constants: the
// y masks (query row t sees rows r >= t of its first group and r <= t of its
// last; every row of the two middle groups) are a few v_cndmask on the packed
// probabilities, and no stage has a per-tile branch.  The three ramp-up groups
// compute only the slots holding a tile; the ramp-down groups compute every
// slot and the emptied ones are discarded.
//
// No softmax reference: a score s (log2 units) has p = 2^s directly, so the
// stage loop has no maximum, no rescaling and no per-tile bias, and the QK
// MFMA starts from the x bias (0 or -inf per key) shared by all slots.  The
// normalisation cancels any common factor of p, so this is exact while p, the
// row sum l and sum(p * v) stay finite and normal: the tile is checked when it
// finishes (l outside [2^-100, inf), NaN, or a non-finite output sum) and such
// tiles are recomputed exactly after the strip by na3d_strip_tile_exact.  Every
// query with its largest score in about [-100, 118] passes; keys more than
// ~26 log2 units below 2^-100 underflow (relative weight below 2^-26 each).
// (gfx950's v_dot2c_f32_bf16 does not keep an fp32 sum: the row sums stay on
// the ones-operand MFMA.)
// LDS bytes of one workgroup of the regular-strip kernel: the K/V ring and the
// staged Q of the next tile.
template <int D, int TX, int RPS, int NBUF, bool ROPE = false>
constexpr int strip_fast_lds_bytes() {
  // ring + staged Q (+ ROPE: each wave's 16 queries' cos and sin rows, 32 pairs of fp32)
  return NBUF * 2 * RPS * ((NA3D_NWX - 1) * TX + 16) * D * 2 + NA3D_NWX * 16 * D * 2 + (ROPE ? NA3D_NWX * 4096 : 0);
}

// `lds`: the workgroup's LDS (strip_fast_lds_bytes), 1 KiB aligned; `id`: its
// work-unit index in [0, sg.total) (as na3d_mfma_body).  LSE: write p.lse (a
// separate instance, so the inference kernels carry none of it).
// ROPE: rotate the queries (p.rc / p.rs tables, head_dim 64, half layout); each tile's
// cos / sin rows are copied into LDS beside its Q.
template <int D, int TX, int RPS, int NBUF, int KY, bool LSE = false, bool ROPE = false>
__device__ __forceinline__ void na3d_strip_fast_body(const Na3dParams p, const Na3dStrips sg, char* lds, int id) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int NWX = NA3D_NWX;
  constexpr int TY = 16 / TX;
  constexpr int NS = (TY + KY - 1) / RPS;  // tile slots per wave: groups a tile's y-union spans
  constexpr int WQX = NWX * TX;           // workgroup query columns
  constexpr int LW = (NWX - 1) * TX + 16; // keys of a row the workgroup reads (no padding)
  constexpr int KPK = 512 / D;            // keys per KiB
  constexpr int RB = LW * D * 2;          // bytes per (tensor, row) region: rows packed back to back
  constexpr int STAGE_B = 2 * RPS * RB;   // K rows 0..RPS-1, then V rows 0..RPS-1
  constexpr int LPT = STAGE_B / 1024 / NWX;  // 1-KiB DMA loads per wave per stage
  constexpr int NRP = RPS / 2;
  constexpr int CPK = D / 8;              // 16-byte chunks per key
  constexpr int KS = D / 32;              // k-steps of the QK MFMA; also 1-KiB loads per wave for 16 query rows
  constexpr int DB = D / 16;
  constexpr int QWB = 16 * D * 2;         // one wave's 16 rows of Q (or of self keys), bytes
  constexpr int QTB = NWX * QWB;          // Q of one tile row of the workgroup
  constexpr int RING_B = NBUF * STAGE_B;
  constexpr int KR = KY / 2;              // window radius in y
  constexpr int FLIP = LW % 8 == 4 ? 1 : 0;  // odd rows start half a swizzle period in: chunk slot bit 2 flips
  constexpr uint32_t LMIN_BITS = (127u - 100u) << 23;  // 2^-100 as an fp32 bit pattern
  constexpr uint32_t INF_BITS = 0x7f800000u;
  static_assert(TY == RPS && TY + KY - 1 == NS * RPS && NS >= 2 && (RPS == 2 || RPS == 4),
                "regular strip geometry: one tile starts per group and its y-union spans NS groups");
  static_assert(D == 64 && (LW % 8 == 4 || LW % 8 == 0), "rows start at a whole or half swizzle period");
  static_assert(LPT * NWX * 1024 == STAGE_B && 2 * LPT * 1024 == RPS * RB,
                "stage layout: waves 0-1 load the K rows, waves 2-3 the V rows, LPT KiB each");
  static_assert(QWB == KS * 1024, "16 query rows are KS 1-KiB loads");
  static_assert(QTB <= RING_B, "tile 0's Q is staged through the ring");

  constexpr int TQB = ROPE ? NWX * 4096 : 0;  // per wave: cos rows of its 16 queries (2 KiB), then sin rows
  static_assert(RING_B + QTB + TQB == strip_fast_lds_bytes<D, TX, RPS, NBUF, ROPE>(), "LDS size");
  static_assert(!ROPE || (D == 64 && TX * TY == 16), "query RoPE: head_dim 64");

  // ---- work unit (as na3d_strip_body) ----
  int t = xcd_tile_order(sg.total, id);
  const int xb = t % sg.nxt;
  t /= sg.nxt;
  const int zt = t % sg.nzt;
  t /= sg.nzt;
  const int ch = t % sg.nch;
  t /= sg.nch;
  const int res = t % sg.nres;
  t /= sg.nres;
  const int h = t % p.H;
  const int b = t / p.H;
  const int dz = p.dil[0], dy = p.dil[1], dx = p.dil[2];
  const int gx = res % dx;
  const int gy = (res / dx) % dy;
  const int gz = res / (dx * dy);

  const int Lz = sub_len(p.L[0], gz, dz);
  const int Lx = sub_len(p.L[2], gx, dx);
  const int qz0 = sub_first(p.org[0], gz, dz), qz1 = sub_end(p.org[0], p.ext[0], gz, dz);
  const int qy0 = sub_first(p.org[1], gy, dy), qy1 = sub_end(p.org[1], p.ext[1], gy, dy);
  const int qx0 = sub_first(p.org[2], gx, dx), qx1 = sub_end(p.org[2], p.ext[2], gx, dx);
  const int iz = qz0 + zt;
  const int ys = qy0 + ch * sg.cty * TY;
  const int ye = min(ys + sg.cty * TY, qy1);
  const int x0 = qx0 + xb * WQX;
  if (iz >= qz1 || ys >= ye || x0 >= qx1) return;  // uniform over the workgroup
  const int NT = (ye - ys + TY - 1) / TY;
  const int S = ys - KR;                 // first key row of tile 0's union (unclamped)
  const int NR = ye - ys + 2 * KR;       // key rows the strip streams
  const int NG = (NR + RPS - 1) / RPS;   // row groups (NT + NS - 1)

  const int kz = p.ker[0], kx = p.ker[2];
  const int sz = win_start(iz, Lz, kz);
  const int X0 = win_start(x0, Lx, kx);

  const int tid = (int)__builtin_amdgcn_workitem_id_x();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int n16 = lane & 15;
  const int g = lane >> 4;
  const int trow = n16 / TX;  // this lane's query row within a tile
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;

  // ---- per-lane x geometry (shared by every tile of the wave) ----
  const int xw0 = x0 + wave * TX;
  const int off_w = win_start(min(xw0, qx1 - 1), Lx, kx) - X0;
  const int qx = xw0 + n16 % TX;
  uint32_t xmask = 0;  // bit i: key 4g+i of the wave's block is outside this lane's x window
  {
    const int sx = win_start(min(qx, qx1 - 1), Lx, kx);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int kxs = X0 + off_w + 4 * g + i;
      xmask |= (kxs >= sx && kxs < sx + kx) ? 0u : (1u << i);
    }
  }

  const int rz = gz + dz * iz;
  const float c2 = p.scale * 1.4426950408889634f;  // scores in log2 units

  // ---- K/V ring lane offsets ----
  // A stage holds RPS rows of LW keys of K, then of V, each key's 16-byte chunks
  // at swizzled slots of the stage-flat key index f = row * LW + x.  Wave w
  // copies the (w & 1)-th half of K (w < 2) or V (w >= 2): LPT 1-KiB loads of
  // 8 keys each, every lane one chunk, at offsets fixed for the whole strip.
  const int64_t rowk = 2 * (int64_t)dy * p.ks[2], rowv = 2 * (int64_t)dy * p.vs[2];
  const bool vwave = wave >= 2;
  const int64_t rowt = vwave ? rowv : rowk;
  const int64_t colt = 2 * (vwave ? p.vs[3] : p.ks[3]);
  uint32_t doff[LPT];
#pragma unroll
  for (int i = 0; i < LPT; ++i) {
    const int f = ((wave & 1) * LPT + i) * KPK + lane / CPK;
    const int row = f / LW, key = f % LW;
    const int c = swz<D>(lane % CPK, f);
    doff[i] = X0 + key < Lx ? (uint32_t)(row * rowt + (int64_t)(gx + dx * (X0 + key)) * colt + 16 * c) : OOB;
  }
  // ---- Q and self-key copies: one (batch, z, head) slice, 31-bit offsets ----
  const u32x4 rq = make_rsrc((const char*)p.q + 2 * ((int64_t)b * p.qs[0] + (int64_t)rz * p.qs[1] + (int64_t)h * p.qs[4]),
                             0x7fffffffu);
  const uint32_t qs2 = (uint32_t)(2 * dy * p.qs[2]);
  uint32_t qxo[KS];
#pragma unroll
  for (int i = 0; i < KS; ++i) {
    const int n = lane / CPK + i * (64 / CPK);
    const int rx = gx + dx * min(xw0 + n % TX, qx1 - 1);
    qxo[i] = (uint32_t)((int64_t)rx * p.qs[3] * 2 + (int64_t)gy * p.qs[2] * 2) + 16 * (lane % CPK);
  }
  // Copy Q of tile j (this wave's 16 queries) to LDS at `off`; ROPE: also the
  // queries' cos and sin rows (128 bytes each; lane l of copy i takes 16 bytes
  // of query 8i + l/8) to this wave's part of the table area.
  const uint32_t tq_lds = lds_base + (uint32_t)(RING_B + QTB) + (uint32_t)wave * 4096;
  auto dma_q = [&](int j, uint32_t off) {
    const int yt0 = ys + TY * j;
    const uint32_t m0 = lds_base + off + (uint32_t)wave * QWB;
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      const int n = lane / CPK + i * (64 / CPK);
      const uint32_t qy = (uint32_t)min(yt0 + n / TX, ye - 1);
      dma_row16(rq, m0 + i * 1024, qxo[i] + qy * qs2);
    }
    if constexpr (ROPE) {
      const u32x4 rc4 = make_rsrc(p.rc, OOB), rs4 = make_rsrc(p.rs, OOB);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int n = lane / 8 + 8 * i;
        const int ry = gy + dy * min(yt0 + n / TX, ye - 1), rx = gx + dx * min(xw0 + n % TX, qx1 - 1);
        const uint32_t o = (uint32_t)(rope_row(p, b, rz, ry, rx) * 128) + 16 * (lane % 8);
        dma_row16(rc4, tq_lds + i * 1024, o);
        dma_row16(rs4, tq_lds + 2048 + i * 1024, o);
      }
    }
  };
  // ---- output: one (batch, z, head) slice ----
  char* obase = (char*)p.o + 2 * ((int64_t)b * p.os[0] + (int64_t)(rz - p.org[0]) * p.os[1] + (int64_t)h * p.os[4]);
  const int64_t orow = 2 * (int64_t)dy * p.os[2];
  const int64_t ooff = 2 * ((int64_t)(gx + dx * qx - p.org[2]) * p.os[3] + (int64_t)(gy - p.org[1]) * p.os[2]) + 8 * g;

  // ---- LDS read offsets of the K/V operands (bytes within row 0 of a stage;
  // row r adds r * RB, and for odd r uses the offsets of chunk bit 2 flipped:
  // entry ks ^ 1 for K, db ^ 2 for V) ----
  uint32_t koff[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int key = off_w + n16;
    koff[ks] = (key * D + 8 * swz<D>(4 * ks + g, key)) * 2;
  }
  uint32_t voffs[DB];
  {
    const int keyv = off_w + 4 * g + (n16 >> 2);
    const int dq = n16 & 3;
#pragma unroll
    for (int db = 0; db < DB; ++db)
      voffs[db] = RPS * RB + (keyv * D + 8 * swz<D>(2 * db + (dq >> 1), keyv) + 4 * (dq & 1)) * 2;
  }

  // ---- tile slots ----
  bf16x8 qreg[NS][KS];
  f32x4 oacc[NS][DB];
  f32x4 lacc[NS];  // row sums (ones x P^T: every row of a column holds the column's sum)
  f32x4 xbias;     // 0 or -inf per key (x window): the C operand of every QK MFMA
#pragma unroll
  for (int i = 0; i < 4; ++i) xbias[i] = ((xmask >> i) & 1) ? -INFINITY : 0.f;
  typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
  bf16x8_t ones = {(bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f};
  // first group: row r (r < RPS - 1) masked for query rows t > r; last group: row r + 1 for t < r + 1
  bool ylo[RPS - 1], yhi[RPS - 1];
#pragma unroll
  for (int r = 0; r < RPS - 1; ++r) {
    ylo[r] = trow > r;
    yhi[r] = trow < r + 1;
  }

  // Tile j enters slot k: Q from LDS, pre-scaled to log2 units.
  auto start_tile = [&](int k, uint32_t off) {
    const char* qb = lds + off + wave * QWB;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qreg[k][ks] = *(const bf16x8*)(qb + n16 * D * 2 + (4 * ks + g) * 16);
    if constexpr (ROPE) {  // pairs 8g .. 8g + 7 of query n16: dims in qreg[k][0], partners in qreg[k][1]
      const char* tb = lds + RING_B + QTB + wave * 4096 + n16 * 128 + g * 32;
      float c[8], sn[8];
      *(f32x4*)&c[0] = *(const f32x4*)(tb);
      *(f32x4*)&c[4] = *(const f32x4*)(tb + 16);
      *(f32x4*)&sn[0] = *(const f32x4*)(tb + 2048);
      *(f32x4*)&sn[4] = *(const f32x4*)(tb + 2048 + 16);
      rope_q_pairs(qreg[k][0], qreg[k][1], c, sn);
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int e = 0; e < 8; ++e) qreg[k][ks][e] = (bf16)((float)qreg[k][ks][e] * c2);
#pragma unroll
    for (int db = 0; db < DB; ++db) oacc[k][db] = (f32x4){0.f, 0.f, 0.f, 0.f};
    lacc[k] = (f32x4){0.f, 0.f, 0.f, 0.f};
  };
  // Normalise and store tile j from slot k; true if the tile needs the exact path.
  auto finish_tile = [&](int k, int j) {
    const float l = lacc[k][0];
    float osum = 0.f;  // infinite or NaN if any output is
#pragma unroll
    for (int db = 0; db < DB; ++db)
      osum += fabsf(oacc[k][db][0]) + fabsf(oacc[k][db][1]) + fabsf(oacc[k][db][2]) + fabsf(oacc[k][db][3]);
    const int qy = ys + TY * j + trow;
    const bool valid = qy < ye && qx < qx1;
    if (valid) {
      // p = 2^s with no reference: the row sum's log2 is the log2-sum-exp itself
      if (LSE && g == 0)
        p.lse[lse_index(p, b, rz - p.org[0], gy + dy * qy - p.org[1], gx + dx * qx - p.org[2], h)] = __log2f(l);
      const float inv = 1.f / l;
      char* op = obase + ooff + (int64_t)qy * orow;
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const u32x2 w = {pack_bf16x2(oacc[k][db][0] * inv, oacc[k][db][1] * inv),
                         pack_bf16x2(oacc[k][db][2] * inv, oacc[k][db][3] * inv)};
        *(u32x2*)(op + 32 * db) = w;
      }
    }
    // l in [2^-100, inf) and a finite output sum (l is never negative: compare the bits)
    const bool ok = __float_as_uint(l) - LMIN_BITS < INF_BITS - LMIN_BITS && __float_as_uint(osum) < INF_BITS;
    return __builtin_amdgcn_ballot_w64(valid && !ok) != 0;
  };

  // QK scores of slot k against the stage's RPS key rows, from the x bias.
  auto scores = [&](int k, const bf16x8 (&ak)[RPS][KS], f32x4 (&sacc)[RPS]) {
#pragma unroll
    for (int r = 0; r < RPS; ++r) {
      sacc[r] = xbias;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        sacc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ak[r][ks], qreg[k][ks], sacc[r], 0, 0, 0);
    }
  };
  // Row sums and O^T += V^T P^T of slot k for the stage's row pairs.
  auto accumulate = [&](int k, const bf16x8 (&pb)[NRP], const bf16x8 (&av)[NRP][DB]) {
#pragma unroll
    for (int rp = 0; rp < NRP; ++rp) {
      lacc[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pb[rp], lacc[k], 0, 0, 0);
#pragma unroll
      for (int db = 0; db < DB; ++db)
        oacc[k][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[rp][db], pb[rp], oacc[k][db], 0, 0, 0);
    }
  };
  auto exp_pack = [&](const f32x4& sv) {
    return (u32x2){pack_bf16x2(__builtin_amdgcn_exp2f(sv[0]), __builtin_amdgcn_exp2f(sv[1])),
                   pack_bf16x2(__builtin_amdgcn_exp2f(sv[2]), __builtin_amdgcn_exp2f(sv[3]))};
  };
  auto rows_to_b = [](const u32x2& a, const u32x2& b) {
    return __builtin_bit_cast(bf16x8, (u32x4){a[0], a[1], b[0], b[1]});
  };

  // One stage's tile math for every slot.  C: slot of the tile in its first group.
  // ACT: bit k set if slot k holds a live tile (ramp groups at a strip's ends skip the others).
  //
  // The tile in its first group (slot C) sees group row r only from query rows
  // t <= r, the tile in its last group (slot C + 1) sees row r only from t >= r:
  // slot C's row r and slot C + 1's row r + 1 are live on disjoint lanes
  // (r < RPS - 1).  When both slots hold tiles their scores on those rows are
  // merged lane by lane before the exponential (one v_exp_f32 per merged value
  // instead of two) and split again by the same masks: for 4-row stages 20
  // exponentials for the two tiles instead of 32, for 2-row stages 12 instead of 16.
  auto stage_math = [&](auto cst, auto act, const bf16x8 (&ak)[RPS][KS], const bf16x8 (&av)[NRP][DB]) {
    constexpr int C = decltype(cst)::value;
    constexpr int ACT = decltype(act)::value;
    constexpr int C1 = (C + 1) % NS;
    constexpr bool MERGE = ((ACT >> C) & 1) && ((ACT >> C1) & 1);
    const u32x2 zero = {0u, 0u};
    if constexpr (MERGE) {
      f32x4 s0[RPS], s1[RPS];
      scores(C, ak, s0);
      scores(C1, ak, s1);
      u32x2 cr[RPS], dr[RPS];  // packed P rows of slot C and of slot C + 1
#pragma unroll
      for (int r = 0; r < RPS - 1; ++r) {
        f32x4 m;
#pragma unroll
        for (int i = 0; i < 4; ++i) m[i] = ylo[r] ? s1[r + 1][i] : s0[r][i];  // t > r: slot C + 1's row r + 1
        const u32x2 pm = exp_pack(m);
        cr[r] = ylo[r] ? zero : pm;      // slot C, row r: t <= r
        dr[r + 1] = yhi[r] ? zero : pm;  // slot C + 1, row r + 1: t >= r + 1
      }
      cr[RPS - 1] = exp_pack(s0[RPS - 1]);
      dr[0] = exp_pack(s1[0]);
      bf16x8 pc[NRP], pd[NRP];
#pragma unroll
      for (int rp = 0; rp < NRP; ++rp) {
        pc[rp] = rows_to_b(cr[2 * rp], cr[2 * rp + 1]);
        pd[rp] = rows_to_b(dr[2 * rp], dr[2 * rp + 1]);
      }
      accumulate(C, pc, av);
      accumulate(C1, pd, av);
    }
#pragma unroll
    for (int tt = MERGE ? 2 : 0; tt < NS; ++tt) {
      const int k = (C + tt) % NS;  // tt = 0: the tile's first group, tt = 1: its last
      if (!((ACT >> k) & 1)) continue;
      f32x4 sacc[RPS];
      scores(k, ak, sacc);
      u32x2 pr[RPS];
#pragma unroll
      for (int r = 0; r < RPS; ++r) {
        pr[r] = exp_pack(sacc[r]);
        if (tt == 0 && r < RPS - 1) pr[r] = ylo[r] ? zero : pr[r];
        if (tt == 1 && r >= 1) pr[r] = yhi[r - 1] ? zero : pr[r];
      }
      bf16x8 pb[NRP];
#pragma unroll
      for (int rp = 0; rp < NRP; ++rp) pb[rp] = rows_to_b(pr[2 * rp], pr[2 * rp + 1]);
      accumulate(k, pb, av);
    }
  };

  // ---- K/V ring over the strip's rows, row-group-major, z-minor ----
  const int64_t zstepk = 2 * (int64_t)dz * p.ks[1], zstepv = 2 * (int64_t)dz * p.vs[1];
  const char* kseg = (const char*)p.k + 2 * ((int64_t)b * p.ks[0] + (int64_t)h * p.ks[4] +
                                             (int64_t)(gz + dz * sz) * p.ks[1] + (int64_t)gy * p.ks[2]) +
                     (int64_t)S * rowk;
  const char* vseg = (const char*)p.v + 2 * ((int64_t)b * p.vs[0] + (int64_t)h * p.vs[4] +
                                             (int64_t)(gz + dz * sz) * p.vs[1] + (int64_t)gy * p.vs[2]) +
                     (int64_t)S * rowv;
  int cz = 0, cp = 0;
  uint32_t issue_off = 0;
  auto issue = [&]() {
    const int nrow = min(max(NR - RPS * cp, 0), RPS);
    const u32x4 rs = vwave ? make_rsrc(vseg + (int64_t)cp * RPS * rowv + (int64_t)cz * zstepv, (uint32_t)(nrow * rowv))
                           : make_rsrc(kseg + (int64_t)cp * RPS * rowk + (int64_t)cz * zstepk, (uint32_t)(nrow * rowk));
    const uint32_t m0 = lds_base + issue_off + (uint32_t)wave * (LPT * 1024);
#pragma unroll
    for (int i = 0; i < LPT; ++i) dma_row16(rs, m0 + i * 1024, doff[i]);
    issue_off = issue_off + STAGE_B == RING_B ? 0 : issue_off + STAGE_B;
    if (++cz == kz) {
      cz = 0;
      ++cp;
    }
  };

  // Tile 0's Q is staged through the ring before the ring starts.
  dma_q(0, 0);
  wait_vmcnt(0);
  start_tile(0, 0);
  wait_lgkm0();
  lds_barrier();  // staged Q read before the ring overwrites it
#pragma unroll
  for (int s = 0; s < NBUF - 1; ++s) issue();

  uint32_t cur_off = 0;
  uint64_t bad_tiles = 0;  // tiles (index < 64) for the exact path
  bool bad_high = false;   // some tile with index >= 64 needs it
  // Group gr (slot gr % NS = C starts tile gr, slot (C + 1) % NS finishes tile gr - NS + 1).
  auto group = [&](auto cst, auto act, int gr) {
    constexpr int C = decltype(cst)::value;
    for (int zc = 0; zc < kz; ++zc) {
      const bool starting = zc == 0 && gr > 0 && gr < NT;
      // The stage read now was issued NBUF - 1 issues ago.  At a tile's start its Q
      // copy (issued after the issue of the group's second slice) must have landed
      // too: only the kz - 2 later issues may still be in flight (none with a
      // two-stage ring: a compile-time wait, no run-time switch at every start).
      if (starting) {
        if constexpr (NBUF == 2)
          wait_vmcnt(0);
        else
          wait_vmcnt((NBUF - 2 < kz - 2 ? NBUF - 2 : kz - 2) * LPT);
      } else
        wait_vmcnt((NBUF - 2) * LPT);
      lds_barrier();
      issue();
      if (starting) start_tile(C, (uint32_t)RING_B);
      // Q of the next group's tile (each wave refills only its own part of the buffer)
      if (zc == 1 && gr + 1 < NT) dma_q(gr + 1, (uint32_t)RING_B);

      asm volatile("" : "+v"(ones));  // keep the ones operand resident
      const char* st = lds + cur_off;
      bf16x8 ak[RPS][KS];
#pragma unroll
      for (int r = 0; r < RPS; ++r)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) ak[r][ks] = *(const bf16x8*)(st + r * RB + koff[ks ^ (FLIP & r)]);
      bf16x8 av[NRP][DB];
#pragma unroll
      for (int rp = 0; rp < NRP; ++rp)
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_PTR(bf16x4, st + voffs[db] + 2 * rp * RB));
          const bf16x4 hi =
              __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_PTR(bf16x4, st + voffs[db ^ (2 * FLIP)] + (2 * rp + 1) * RB));
          av[rp][db] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
      stage_math(cst, act, ak, av);
      cur_off = cur_off + STAGE_B == RING_B ? 0 : cur_off + STAGE_B;
    }
    const int jf = gr - (NS - 1);
    if (jf >= 0 && jf < NT && finish_tile((C + 1) % NS, jf)) {
      if (jf < 64)
        bad_tiles |= 1ull << jf;
      else
        bad_high = true;
    }
  };
  using ALL = std::integral_constant<int, (1 << NS) - 1>;
  // Ramp-up: tile g starts in group g (slot g), so groups 0 .. NS-2 compute
  // only the slots already holding a tile.  From group NS-1 on every slot
  // computes (the ramp-down's emptied slots too: separate instances for the
  // ramp-down groups make the register allocator spill).
  static_for<NS - 1>([&](auto ig) {
    constexpr int G = decltype(ig)::value;
    group(std::integral_constant<int, G>{}, std::integral_constant<int, (1 << (G + 1)) - 1>{}, G);
  });
  for (int gr = NS - 1;; gr += NS) {  // NG = NT + NS - 1 >= NS
    bool done = false;
    static_for<NS>([&](auto ii) {
      constexpr int I = decltype(ii)::value;
      if (!done) {
        group(std::integral_constant<int, (NS - 1 + I) % NS>{}, ALL{}, gr + I);
        done = gr + I + 1 >= NG;
      }
    });
    if (done) break;
  }
  wait_vmcnt(0);  // the ring's trailing (empty) stages

  // Rare: tiles whose sums left the range the reference-free softmax keeps
  // exact, recomputed after the strip (their stores above are overwritten).
  if (bad_tiles != 0 || bad_high) {
    __builtin_amdgcn_s_waitcnt(0);
    for (int j = 0; j < NT; ++j)
      if (j < 64 ? ((bad_tiles >> j) & 1) : bad_high)
        na3d_strip_tile_exact<TX, ROPE>(&p, StripTile{b, h, gz, gy, gx, iz, ys + TY * j, ye, xw0, qx1});
  }
#endif
}

// Two workgroups per CU (the 13-row window: 64 KiB of LDS each, ~230 VGPRs);
// three for 5-row windows (48 KiB of LDS, 163 VGPRs; wider windows would spill).
template <int D, int TX, int RPS, int NBUF, int KY, bool LSE>
__global__ __launch_bounds__(256, TX == 8 && KY <= 5 ? 3 : 2) void na3d_strip_fast_kernel(Na3dParams p, Na3dStrips sg) {
  __shared__ __attribute__((aligned(1024))) char lds[strip_fast_lds_bytes<D, TX, RPS, NBUF>()];
  na3d_strip_fast_body<D, TX, RPS, NBUF, KY, LSE>(p, sg, lds, (int)__builtin_amdgcn_workgroup_id_x());
}

// Small windows in one launch: the regular strips of the rows whose y window is
// not clamped, and the general kernel (a 2-stage ring, workgroups as tall as an
// edge: 2 rows for ky = 5, else 4) over the clamped rows at each end, so the short
// edge workgroups fill the strips' tail instead of running after them.  Workgroup
// ids [0, n0) take the strips, [n0, n0 + n1) the top edge, the rest the bottom
// edge; n0 and n1 are multiples of 8, so each part keeps its XCD-aware tile order.
// Ring depth of the strips: three stages for ky 7 and 9 without the query rotation
// (68 KiB of LDS, still two workgroups per CU; configs[3] plain 0.343 -> 0.328 ms,
// configs[1] 0.088 -> 0.086 ms); two where a third stage would cost occupancy (ky 5
// runs three workgroups per CU at 48 KiB; the rotation's tables take another 16 KiB).
template <int KY, bool LSE, bool ROPE = false, int NBUF = (ROPE || KY <= 5) ? 2 : 3>
__global__ __launch_bounds__(256, KY <= 5 ? 3 : 2) void na3d_small_fused_kernel(Na3dParams mid, Na3dStrips sg,
                                                                               Na3dParams e0, Na3dTiles t0,
                                                                               Na3dParams e1, Na3dTiles t1, int n0,
                                                                               int n1) {
  constexpr int NTYE = KY <= 5 ? 1 : 2;
  constexpr int LS = strip_fast_lds_bytes<64, 8, 2, NBUF, ROPE>(), LE = mfma_lds_bytes<64, 8, 2, 2>();
  __shared__ __attribute__((aligned(1024))) char lds[LS > LE ? LS : LE];
  const int id = (int)__builtin_amdgcn_workgroup_id_x();
  if (id < n0) {
    if (id < sg.total) na3d_strip_fast_body<64, 8, 2, NBUF, KY, LSE, ROPE>(mid, sg, lds, id);
  } else if (id < n0 + n1) {
    if (id - n0 < t0.total) na3d_mfma_body<64, 8, NTYE, 2, 2, ROPE>(e0, t0, lds, id - n0);
  } else if (id - n0 - n1 < t1.total) {
    na3d_mfma_body<64, 8, NTYE, 2, 2, ROPE>(e1, t1, lds, id - n0 - n1);
  }
}


// ---------------------------------------------------------------------------
// Small windows on query regions (na3d_region_kernel): kz = 3, ky = KY, kx <= KY (odd),
// head_dim 64, bf16; any dilation and query box.  The template covers KY in {3, 5, 7};
// the host takes it for ky = 3 (region_fits), where it beats the strips.
//
// A workgroup of 8 waves owns a region of 8 query rows x 16 query columns of one
// (batch, head, dilation residue) at every query z of the box, and walks the key
// z-slices those queries' windows reach once, in order.  Stage s copies the
// (7 + KY) x (15 + KY) keys of slice s that any window of the region can touch
// (K, then V; keys past the grid read as zero) into an LDS ring (three stages where
// they fit, else two), so a K/V slice crosses L2 -> LDS once per region instead of
// once per query z.  The copies of a stage are issued a share per row pair during
// the stage before it, beside the MFMAs, not in one burst after the barrier (one
// workgroup per CU: every wave reaches the barrier together).  Wave w owns the
// 2 x 8 tile at rows 2 (w >> 1), columns 8 (w & 1) of the region at every z: the
// tile of query z zq lives in register slot (zq - zbase) & 3 during the three stages
// whose slice its z window holds (at most four tiles overlap, at the clamped z ends;
// three in the interior, where the stage loop, unrolled four times, knows the live
// slots at compile time).  Per stage a wave reads each of its tile's KY + 1 key rows
// (one 16-key block: the tile's 8 + kx - 1 columns) once and feeds every live slot.
// Rows 1 .. KY - 1 of a tile's union lie in both query rows' windows; rows 0 and KY
// are complementary (query row 0 always takes row 0; query row 1 takes exactly one
// of them), so they form one PV step and share one exponential.  Every clamped edge
// (z, y and x) is a mask: there is no separate edge kernel.  Softmax as the strip
// kernels: p = 2^s of the log2-unit scores, the x window as the QK MFMA's C operand,
// row sums by a ones-operand MFMA, a range check per tile and an exact recompute of
// the rare tiles that leave the range.
// ---------------------------------------------------------------------------
struct Na3dRegions {
  int nrx, nry;  // regions per (batch, head, residue) along x and along y
  int nres;      // dil_z * dil_y * dil_x
  int total;     // workgroups
};

template <int KY>
struct RegionGeom {
  static constexpr int NRY = 7 + KY;                 // key rows a region's windows reach
  static constexpr int LW = 15 + KY;                 // keys per row (kx <= KY)
  static constexpr int NK = (NRY * LW + 7) / 8 * 8;  // keys per tensor, whole 1-KiB copies
  static constexpr int REG_B = NK * 128;             // bytes of one tensor's keys (head_dim 64)
  static constexpr int STAGE_B = 2 * REG_B;          // K, then V
  static constexpr int NDMA = 2 * NK / 8;            // 1-KiB copies per stage
  static constexpr int DPW = (NDMA + 7) / 8;         // per wave (copy 8 j + wave)
  static constexpr int IDLE_B = (8 * DPW - NDMA) * 1024;   // where the waves' idle copies land
  static constexpr int NBUF = 3 * STAGE_B + IDLE_B <= 160 * 1024 ? 3 : 2;  // ring stages: three where they fit
  static constexpr int LDS_B = NBUF * STAGE_B + IDLE_B;
  static_assert(LDS_B <= 160 * 1024, "the ring fits the CU's LDS");
};

template <int KY, bool LSE, bool ROPE>
__global__ __launch_bounds__(512, 1) void na3d_region_kernel(Na3dParams p, Na3dRegions rg) {
#if defined(__HIP_DEVICE_COMPILE__)
  using G = RegionGeom<KY>;
  constexpr int LW = G::LW, NRY = G::NRY, REG_B = G::REG_B, STAGE_B = G::STAGE_B, NDMA = G::NDMA, DPW = G::DPW;
  constexpr int NP = (KY + 1) / 2;  // PV steps of a tile: row pairs (0, KY), (1, 2), (3, 4), ...
  constexpr int RB = LW * 128;      // bytes of one region row (a multiple of 256: rows keep the bank pattern)
  constexpr uint32_t LMIN_BITS = (127u - 100u) << 23;  // 2^-100
  constexpr uint32_t INF_BITS = 0x7f800000u;
  static_assert(RB % 256 == 0, "row starts keep the chunk swizzle conflict-free");
  __shared__ __attribute__((aligned(1024))) char lds[G::LDS_B];

  // ---- work unit: (batch, head, residue, region y, region x), x fastest ----
  int t = xcd_tile_order(rg.total, (int)__builtin_amdgcn_workgroup_id_x());
  const int rx = t % rg.nrx;
  t /= rg.nrx;
  const int ry = t % rg.nry;
  t /= rg.nry;
  const int res = t % rg.nres;
  t /= rg.nres;
  const int h = t % p.H;
  const int b = t / p.H;
  const int dz = p.dil[0], dy = p.dil[1], dx = p.dil[2];
  const int gx = res % dx, gy = (res / dx) % dy, gz = res / (dx * dy);
  const int Lz = sub_len(p.L[0], gz, dz), Ly = sub_len(p.L[1], gy, dy), Lx = sub_len(p.L[2], gx, dx);
  const int qz0 = sub_first(p.org[0], gz, dz), qz1 = sub_end(p.org[0], p.ext[0], gz, dz);
  const int qy0 = sub_first(p.org[1], gy, dy), qy1 = sub_end(p.org[1], p.ext[1], gy, dy);
  const int qx0 = sub_first(p.org[2], gx, dx), qx1 = sub_end(p.org[2], p.ext[2], gx, dx);
  const int y0 = qy0 + 8 * ry, x0 = qx0 + 16 * rx;
  if (qz0 >= qz1 || y0 >= qy1 || x0 >= qx1) return;  // uniform over the workgroup
  const int kz = p.ker[0], kx = p.ker[2];
  const int RY0 = win_start(y0, Ly, KY), RX0 = win_start(x0, Lx, kx);  // the region's first key row / column

  const int tid = (int)__builtin_amdgcn_workitem_id_x();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, n16 = lane & 15, g = lane >> 4;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;

  // ---- this wave's tile: query rows yt, yt + 1, columns xt .. xt + 7 ----
  const int yt = y0 + 2 * (wave >> 1), xt = x0 + 8 * (wave & 1);
  const int by = win_start(min(yt, qy1 - 1), Ly, KY) - RY0;  // the tile's first union row in the region (<= 6)
  // first region column of the tile's 16-key block: its 8 + kx - 1 columns start at
  // or after it and end inside the region's LW
  const int bx = (wave & 1) ? min(win_start(min(xt, qx1 - 1), Lx, kx) - RX0, LW - 16) : 0;
  const int tq = n16 >> 3;  // this lane's query: row tq, column n16 & 7 of the tile
  const int qyc = min(yt + tq, qy1 - 1), qxc = min(xt + (n16 & 7), qx1 - 1);
  const bool qvalid = yt + tq < qy1 && xt + (n16 & 7) < qx1;
  // the lane's y window covers union rows [d, d + KY), d in {0, 1}: d = 1 means row KY, not row 0
  const bool rowky = win_start(qyc, Ly, KY) - RY0 - by == 1;
  f32x4 xbias;  // 0 or -inf for keys bx + 4g + i of the block (x window): the QK MFMA's C operand
  {
    const int sx = win_start(qxc, Lx, kx);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int kc = RX0 + bx + 4 * g + i;
      xbias[i] = (kc >= sx && kc < sx + kx) ? 0.f : -INFINITY;
    }
  }

  // ---- LDS read offsets within a stage (row r of the tile's union adds r * RB);
  // chunk c of the key in region column col sits at slot c ^ (col & 7) ----
  uint32_t koff[2], voff[4];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const int col = bx + n16;
    koff[ks] = (uint32_t)(by * RB + col * 128 + 16 * ((4 * ks + g) ^ (col & 7)));
  }
  {
    const int col = bx + 4 * g + (n16 >> 2), dq = n16 & 3;
#pragma unroll
    for (int db = 0; db < 4; ++db)
      voff[db] = (uint32_t)(REG_B + by * RB + col * 128 + 16 * ((2 * db + (dq >> 1)) ^ (col & 7)) + 8 * (dq & 1));
  }

  // ---- copies: stage copy J = 8 j + wave (J < NDMA / 2: K keys 8J .. 8J + 7 of the
  // region, row-major; else the same keys of V); lane l fills slot l & 7 of key l / 8 ----
  const int64_t rowk = 2 * (int64_t)dy * p.ks[2], rowv = 2 * (int64_t)dy * p.vs[2];
  uint32_t doff[DPW];
#pragma unroll
  for (int j = 0; j < DPW; ++j) {
    const int J = 8 * j + wave;
    const bool isv = J >= NDMA / 2;
    const int f = 8 * (isv ? J - NDMA / 2 : J) + lane / 8;
    const int row = f / LW, col = f % LW;
    const bool ok = J < NDMA && f < NRY * LW && RY0 + row < Ly && RX0 + col < Lx;
    const int64_t o = row * (isv ? rowv : rowk) + (int64_t)(gx + dx * (RX0 + col)) * 2 * (isv ? p.vs[3] : p.ks[3]) +
                      16 * ((lane & 7) ^ (col & 7));
    doff[j] = ok ? (uint32_t)o : OOB;
  }
  const char* kbase = (const char*)p.k + 2 * ((int64_t)b * p.ks[0] + (int64_t)h * p.ks[4] + (int64_t)gz * p.ks[1] +
                                              (int64_t)(gy + dy * RY0) * p.ks[2]);
  const char* vbase = (const char*)p.v + 2 * ((int64_t)b * p.vs[0] + (int64_t)h * p.vs[4] + (int64_t)gz * p.vs[1] +
                                              (int64_t)(gy + dy * RY0) * p.vs[2]);
  const int64_t zk = 2 * (int64_t)dz * p.ks[1], zv = 2 * (int64_t)dz * p.vs[1];
  // Copies j in [J0, J1) of the wave into the ring slot at byte `slot`, from the K and V
  // descriptors of one slice.  Copy J >= NDMA (the last of some waves) reads zeros into
  // the idle area past the ring, so no copy sits under a branch.
  uint32_t ddst[DPW];  // destination of copy j within a slot (or the idle area, minus the slot)
#pragma unroll
  for (int j = 0; j < DPW; ++j) {
    const int J = 8 * j + wave;
    ddst[j] = J >= NDMA ? 0u : (uint32_t)(J >= NDMA / 2 ? REG_B + 1024 * (J - NDMA / 2) : 1024 * J);
    if (J >= NDMA) doff[j] = OOB;
  }
  const uint32_t idle_dst = lds_base + (uint32_t)(G::NBUF * STAGE_B) + 1024u * (uint32_t)max(0, 8 * (DPW - 1) + wave - NDMA);
  auto issue_part = [&](const u32x4& rk, const u32x4& rv, uint32_t slot, auto j0c, auto j1c) {
    constexpr int J0 = decltype(j0c)::value, J1 = decltype(j1c)::value;
    static_for<DPW>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      if constexpr (j >= J0 && j < J1) {
        const int J = 8 * j + wave;  // uniform
        const bool isv = J >= NDMA / 2;
        dma_row16(isv ? rv : rk, J >= NDMA ? idle_dst : lds_base + slot + ddst[j], doff[j]);
      }
    });
  };
  auto issue = [&](int s, uint32_t slot) {
    const u32x4 rk = make_rsrc(kbase + s * zk, OOB), rv = make_rsrc(vbase + s * zv, OOB);
    issue_part(rk, rv, slot, std::integral_constant<int, 0>{}, std::integral_constant<int, DPW>{});
  };

  // ---- queries: lane (row tq, column n16 & 7) loads dims 8g .. 8g + 7 and 32 + 8g .. 32 + 8g + 7 ----
  const char* qlane = (const char*)p.q + 2 * ((int64_t)b * p.qs[0] + (int64_t)h * p.qs[4] + (int64_t)gz * p.qs[1] +
                                              (int64_t)(gy + dy * qyc) * p.qs[2] + (int64_t)(gx + dx * qxc) * p.qs[3]);
  const int64_t qzs = 2 * (int64_t)dz * p.qs[1];
  auto load_q = [&](int zq, bf16x8 (&qv)[2]) {
    const char* a = qlane + zq * qzs;
    qv[0] = *(const bf16x8*)(a + 16 * g);
    qv[1] = *(const bf16x8*)(a + 64 + 16 * g);
  };
  // ROPE: cos / sin of pairs 8g .. 8g + 7 (half layout: dims j and j + 32) of the lane's query
  auto load_rope = [&](int zq, f32x4 (&c)[2], f32x4 (&sn)[2]) {
    if constexpr (ROPE) {
      const int64_t r = rope_row(p, b, gz + dz * zq, gy + dy * qyc, gx + dx * qxc) * 32 + 8 * g;
      c[0] = *(const f32x4*)(p.rc + r);
      c[1] = *(const f32x4*)(p.rc + r + 4);
      sn[0] = *(const f32x4*)(p.rs + r);
      sn[1] = *(const f32x4*)(p.rs + r + 4);
    }
  };
  char* olane = (char*)p.o + 2 * ((int64_t)b * p.os[0] + (int64_t)h * p.os[4] + (int64_t)(gz - p.org[0]) * p.os[1] +
                                  (int64_t)(gy + dy * qyc - p.org[1]) * p.os[2] +
                                  (int64_t)(gx + dx * qxc - p.org[2]) * p.os[3]) +
                8 * g;
  const int64_t ozs = 2 * (int64_t)dz * p.os[1];
  const float c2 = p.scale * 1.4426950408889634f;  // scores in log2 units

  // ---- tile slots ----
  bf16x8 qreg[4][2];
  f32x4 oacc[4][4];
  f32x4 lacc[4];
  typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
  bf16x8_t ones = {(bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f};
  // A tile enters slot k: its queries (rotated with ROPE) pre-scaled to log2 units.
  auto start = [&](auto kc, const bf16x8 (&qv)[2], const f32x4 (&c)[2], const f32x4 (&sn)[2]) {
    constexpr int k = decltype(kc)::value;
    bf16x8 lo = qv[0], hi = qv[1];
    if constexpr (ROPE) {
      float cc[8], ss[8];
      *(f32x4*)&cc[0] = c[0];
      *(f32x4*)&cc[4] = c[1];
      *(f32x4*)&ss[0] = sn[0];
      *(f32x4*)&ss[4] = sn[1];
      rope_q_pairs(lo, hi, cc, ss);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      qreg[k][0][e] = (bf16)((float)lo[e] * c2);
      qreg[k][1][e] = (bf16)((float)hi[e] * c2);
    }
#pragma unroll
    for (int db = 0; db < 4; ++db) oacc[k][db] = (f32x4){0.f, 0.f, 0.f, 0.f};
    lacc[k] = (f32x4){0.f, 0.f, 0.f, 0.f};
  };

  // Deferred output of one finished tile: stored at the next stage's start, after
  // that stage's copies are issued, so the stage-start wait does not cover a
  // store issued just before it.
  u32x2 pend[4];
  char* pend_ptr = nullptr;
  float pend_lse = 0.f;
  float* pend_lse_ptr = nullptr;
  bool pend_on = false;  // uniform
  auto flush = [&]() {
    if (pend_on) {
      if (qvalid) {
#pragma unroll
        for (int db = 0; db < 4; ++db) *(u32x2*)(pend_ptr + 32 * db) = pend[db];
        if (LSE && g == 0) *pend_lse_ptr = pend_lse;
      }
      pend_on = false;
    }
  };
  // Normalise slot k's tile (query z zq); true if it needs the exact path.
  auto finish = [&](auto kc, int zq) {
    constexpr int k = decltype(kc)::value;
    const float l = lacc[k][0];
    float osum = 0.f;
#pragma unroll
    for (int db = 0; db < 4; ++db)
      osum += fabsf(oacc[k][db][0]) + fabsf(oacc[k][db][1]) + fabsf(oacc[k][db][2]) + fabsf(oacc[k][db][3]);
    const float inv = 1.f / l;
    u32x2 w[4];
#pragma unroll
    for (int db = 0; db < 4; ++db)
      w[db] = (u32x2){pack_bf16x2(oacc[k][db][0] * inv, oacc[k][db][1] * inv),
                      pack_bf16x2(oacc[k][db][2] * inv, oacc[k][db][3] * inv)};
    char* op = olane + zq * ozs;
    float* lp = nullptr;
    if (LSE) lp = p.lse + lse_index(p, b, gz + dz * zq - p.org[0], gy + dy * qyc - p.org[1], gx + dx * qxc - p.org[2], h);
    if (!pend_on) {
#pragma unroll
      for (int db = 0; db < 4; ++db) pend[db] = w[db];
      pend_ptr = op;
      pend_lse = __log2f(l);
      pend_lse_ptr = lp;
      pend_on = true;
    } else if (qvalid) {  // a second tile in one stage (the clamped z ends): store now
#pragma unroll
      for (int db = 0; db < 4; ++db) *(u32x2*)(op + 32 * db) = w[db];
      if (LSE && g == 0) *lp = __log2f(l);
    }
    const bool ok = __float_as_uint(l) - LMIN_BITS < INF_BITS - LMIN_BITS && __float_as_uint(osum) < INF_BITS;
    return __builtin_amdgcn_ballot_w64(qvalid && !ok) != 0;
  };

  auto exp_pack = [&](const f32x4& sv) {
    return (u32x2){pack_bf16x2(__builtin_amdgcn_exp2f(sv[0]), __builtin_amdgcn_exp2f(sv[1])),
                   pack_bf16x2(__builtin_amdgcn_exp2f(sv[2]), __builtin_amdgcn_exp2f(sv[3]))};
  };
  // One stage's math on the slots in ACT (a compile-time mask; 0xF at the z ends,
  // where inactive slots compute into accumulators their next tile resets).
  // hook(pc) runs after pair pc's operand reads (the stage's copies go out there, a
  // share per pair, so the CU's address path streams them beside the MFMAs rather
  // than in one burst after the barrier).
  auto stage_math = [&](auto actc, uint32_t cur, auto&& hook) {
    constexpr int ACT = decltype(actc)::value;
    const char* st = lds + cur;
    asm volatile("" : "+v"(ones));  // keep the ones operand resident
    static_for<NP>([&](auto pc) {
      constexpr int PI = decltype(pc)::value;
      constexpr int RA = PI == 0 ? 0 : 2 * PI - 1, RBW = PI == 0 ? KY : 2 * PI;
      bf16x8 ak[2][2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        ak[0][ks] = *(const bf16x8*)(st + RA * RB + koff[ks]);
        ak[1][ks] = *(const bf16x8*)(st + RBW * RB + koff[ks]);
      }
      bf16x8 av[4];
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_PTR(bf16x4, st + voff[db] + RA * RB));
        const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_PTR(bf16x4, st + voff[db] + RBW * RB));
        av[db] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      }
      hook(pc);
      f32x4 sc[4][2];  // every live slot's scores first, so the exponentials wait on none of them
      static_for<4>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        if constexpr ((ACT >> k) & 1) {
          sc[k][0] = xbias;
          sc[k][1] = xbias;
#pragma unroll
          for (int ks = 0; ks < 2; ++ks) {
            sc[k][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ak[0][ks], qreg[k][ks], sc[k][0], 0, 0, 0);
            sc[k][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ak[1][ks], qreg[k][ks], sc[k][1], 0, 0, 0);
          }
        }
      });
      static_for<4>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        if constexpr ((ACT >> k) & 1) {
          const f32x4 sa = sc[k][0], sb = sc[k][1];
          u32x2 pa, pb;
          if constexpr (PI == 0) {  // rows 0 and KY: one exponential, split by the lane's y window
            f32x4 m;
#pragma unroll
            for (int i = 0; i < 4; ++i) m[i] = rowky ? sb[i] : sa[i];
            const u32x2 pm = exp_pack(m), zero = {0u, 0u};
            pa = rowky ? zero : pm;
            pb = rowky ? pm : zero;
          } else {
            pa = exp_pack(sa);
            pb = exp_pack(sb);
          }
          const bf16x8 pp = __builtin_bit_cast(bf16x8, (u32x4){pa[0], pa[1], pb[0], pb[1]});
          lacc[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pp, lacc[k], 0, 0, 0);
#pragma unroll
          for (int db = 0; db < 4; ++db)
            oacc[k][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[db], pp, oacc[k][db], 0, 0, 0);
        }
      });
    });
  };

  // ---- the z walk: slices [S0, S1); the tiles live at stage s are zq in [zlo(s), zhi(s)]:
  // zq = s - 1, s, s + 1 in the interior, plus s - 2 or s + 2 at the clamped z ends (at
  // most four: the host checks).  The tile of query z zq holds slot (zq - zbase) & 3, so
  // in the stage loop unrolled four times the interior slots are compile-time. ----
  constexpr int H2 = 1;  // kz / 2 (kz = 3)
  const int S0 = win_start(qz0, Lz, kz), S1 = win_start(qz1 - 1, Lz, kz) + kz;
  const int zbase = S0 - 1;
  auto zhi_of = [&](int s) { return s >= Lz - kz ? qz1 - 1 : min(qz1 - 1, s + H2); };
  auto zlo_of = [&](int s) { return s - kz + 1 <= 0 ? qz0 : max(qz0, s - kz + 1 + H2); };
  auto zstart = [&](int zq) { return win_start(zq, Lz, kz); };
  auto slot_z = [&](int k, int zl) { return zl + ((k + zbase - zl) & 3); };  // the zq >= zl slot k holds

  // Ring: stage s in slot (s - S0) % NBUF; stage s issues stage s + NBUF - 1 into the slot
  // that stage s - 1 read (free once every wave has passed stage s's barrier).
  constexpr int NBUF = G::NBUF;
  issue(S0, 0);
  if (NBUF == 3 && S0 + 1 < S1) issue(S0 + 1, STAGE_B);
  {  // the tiles of the first slice: loaded here
    const int zl = zlo_of(S0), zh = zhi_of(S0);
    static_for<4>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      const int zq = slot_z(k, zl);
      if (zq <= zh) {
        bf16x8 qv[2];
        f32x4 c[2], sn[2];
        load_q(zq, qv);
        load_rope(zq, c, sn);
        start(kc, qv, c, sn);
      }
    });
  }
  // Prefetch of the next stage's first tile (with ROPE: its tables too); a second
  // tile that starts in the same stage (the clamped z ends) loads at its start.
  bf16x8 qpre[2];
  f32x4 cpre[2], spre[2];
  int pf_z = 1 << 30;  // query z of the prefetched tile (uniform)
  auto prefetch = [&](int s) {  // the first tile starting at stage s, if any
    const int zq = zhi_of(s - 1) + 1;
    pf_z = 1 << 30;
    if (s < S1 && zq <= zhi_of(s)) {
      load_q(zq, qpre);
      load_rope(zq, cpre, spre);
      pf_z = zq;
    }
  };

  uint64_t bad_lo = 0;  // tiles (zq < 64) for the exact path
  bool bad_hi = false;
  uint32_t cur = 0, wr = (NBUF - 1) * STAGE_B;
  auto next_slot = [](uint32_t o) { return o + STAGE_B == NBUF * STAGE_B ? 0u : o + STAGE_B; };
  for (int s4 = S0; s4 < S1; s4 += 4) {
    static_for<4>([&](auto ic) {
      constexpr int I = decltype(ic)::value;
      constexpr int IDLE = (I + 3) & 3;  // the slot of zq = s +- 2 (stage s = s4 + I)
      const int s = s4 + I;
      if (s < S1) {
        // Stage s's copies and the prefetched queries have landed once at most the copies
        // of stage s + 1 (issued after them; loads complete in order) are outstanding.
        if (NBUF == 3 && s > S0)
          wait_vmcnt(DPW);
        else
          wait_vmcnt(0);
        lds_barrier();  // every wave's copies of stage s have landed; slot wr is free
        // the stage this one issues: past the walk's end the last slice again, into a slot
        // nobody reads (the walk's last wait drains those copies)
        const int sn = min(s + NBUF - 1, S1 - 1);
        const u32x4 rk = make_rsrc(kbase + sn * zk, OOB), rv = make_rsrc(vbase + sn * zv, OOB);
        flush();
        const int zl = zlo_of(s), zh = zhi_of(s);
        if (s > S0) {  // tiles starting at s: zq in (zhi(s - 1), zh]
          static_for<4>([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            const int zq = slot_z(k, zl);
            if (zq <= zh && zstart(zq) == s) {
              if (zq == pf_z) {
                start(kc, qpre, cpre, spre);
              } else {
                bf16x8 qv[2];
                f32x4 c[2], sn[2];
                load_q(zq, qv);
                load_rope(zq, c, sn);
                start(kc, qv, c, sn);
              }
            }
          });
        }
        prefetch(s + 1);
        // slots of zq = s - 1, s, s + 1 (an idle one computes into accumulators its next tile resets)
        stage_math(std::integral_constant<int, 0xF & ~(1 << IDLE)>{}, cur, [&](auto pc) {
          constexpr int PI = decltype(pc)::value;
          issue_part(rk, rv, wr, std::integral_constant<int, PI * DPW / NP>{},
                     std::integral_constant<int, (PI + 1) * DPW / NP>{});
        });
        if (zl <= s - 2 || zh >= s + 2) stage_math(std::integral_constant<int, 1 << IDLE>{}, cur, [](auto) {});
        static_for<4>([&](auto kc) {
          constexpr int k = decltype(kc)::value;
          const int zq = slot_z(k, zl);
          if (zq <= zh && zstart(zq) + kz - 1 == s && finish(kc, zq)) {
            if (zq < 64)
              bad_lo |= 1ull << zq;
            else
              bad_hi = true;
          }
        });
        cur = next_slot(cur);
        wr = next_slot(wr);
      }
    });
  }
  wait_vmcnt(0);  // the copies issued past the walk's end land before the workgroup's LDS is released
  flush();
  if (bad_lo != 0 || bad_hi) {
    __builtin_amdgcn_s_waitcnt(0);
    for (int zq = qz0; zq < qz1; ++zq)
      if (zq < 64 ? ((bad_lo >> zq) & 1) : bad_hi)
        na3d_strip_tile_exact<8, ROPE>(&p, StripTile{b, h, gz, gy, gx, zq, yt, qy1, xt, qx1});
  }
#endif
}

// ---------------------------------------------------------------------------
// Depth-wise (column) attention: window (Z, 1, 1) over the whole z axis, Z <= 32,
// head_dim 64, bf16, the whole grid as the query box.  Every token attends the Z
// tokens of its own (y, x) column; the tile kernels above would compute a 16 x 16
// score block per 16 useful pairs here.
//
// One wave per (batch, y, x, head) column, four per workgroup (consecutive heads
// of one column: their rows are 128 bytes apart).  The column's Q, K and V rows
// are loaded with whole-line loads (lane l: row l / 8 + 8 c, 16-byte chunk l % 8;
// rows past Z zero) and pass in turn through the wave's 4 KiB of LDS (chunk slot
// (l % 8) ^ (row % 8)) into the MFMA layouts.  S^T = K Q^T on v_mfma_f32_32x32x16_bf16 (keys on M, queries
// on N, Z padded to 32); the softmax runs over a lane's 16 keys and its partner
// lane's (l ^ 32) other 16.  O^T = V^T P^T: P^T comes from the score lanes as they
// are (k-index 8 hi + m of k-step t is key 16 t + 4 hi + m for m < 4 and
// 16 t + 8 + 4 hi + m - 4 otherwise, the keys the score layout gives lane half hi),
// and V^T gathers the same keys' values of one dimension from LDS.  Lane
// (query n, hi) ends holding O^T rows 32 db + 8 i + 4 hi + e, four consecutive dims
// that it writes to the buffer's row n, read back and stored as whole rows.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void na3d_column_kernel(Na3dParams p, int64_t items) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __attribute__((aligned(16))) bf16 sh[4][32 * 64];  // per wave: Q, then K, then V rows
  const int tid = (int)__builtin_amdgcn_workitem_id_x();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int64_t item = (int64_t)__builtin_amdgcn_workgroup_id_x() * 4 + wave;
  if (item >= items) return;  // uniform over the wave; no barrier below
  int64_t t = item;
  const int h = (int)(t % p.H);
  t /= p.H;
  const int x = (int)(t % p.L[2]);
  t /= p.L[2];
  const int y = (int)(t % p.L[1]);
  const int b = (int)(t / p.L[1]);
  const int Z = p.L[0];
  const int n = lane & 31, hi = lane >> 5;
  const bf16* src[3] = {
      (const bf16*)p.q + (int64_t)b * p.qs[0] + (int64_t)y * p.qs[2] + (int64_t)x * p.qs[3] + (int64_t)h * p.qs[4],
      (const bf16*)p.k + (int64_t)b * p.ks[0] + (int64_t)y * p.ks[2] + (int64_t)x * p.ks[3] + (int64_t)h * p.ks[4],
      (const bf16*)p.v + (int64_t)b * p.vs[0] + (int64_t)y * p.vs[2] + (int64_t)x * p.vs[3] + (int64_t)h * p.vs[4]};
  const int64_t zs[3] = {p.qs[1], p.ks[1], p.vs[1]};
  bf16* const sw = sh[wave];
  // element (row r, dim d) of the staged tensor
  auto at = [](int r, int d) { return r * 64 + 8 * ((d >> 3) ^ (r & 7)) + (d & 7); };

  u32x4 w[3][4];  // all three tensors' loads in flight at once
#pragma unroll
  for (int tt = 0; tt < 3; ++tt)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int r = lane / 8 + 8 * c;
      w[tt][c] = (u32x4){0u, 0u, 0u, 0u};
      if (r < Z) w[tt][c] = *(const u32x4*)(src[tt] + (int64_t)r * zs[tt] + 8 * (lane % 8));
    }
  // Through the wave's one LDS buffer in turn (its own rows only: no barrier); the
  // waits order each tensor's fragment reads before the next tensor's writes.
  auto stage = [&](int tt) {
    wait_lgkm0();
#pragma unroll
    for (int c = 0; c < 4; ++c) *(u32x4*)&sw[at(lane / 8 + 8 * c, 8 * (lane % 8))] = w[tt][c];
    wait_lgkm0();
  };
  bf16x8 qf[4], kf[4];
  stage(0);
#pragma unroll
  for (int st = 0; st < 4; ++st) qf[st] = *(const bf16x8*)&sw[at(n, 16 * st + 8 * hi)];
  stage(1);
#pragma unroll
  for (int st = 0; st < 4; ++st) kf[st] = *(const bf16x8*)&sw[at(n, 16 * st + 8 * hi)];
  stage(2);
  // Scores S^T[key][query], log2 units.
  f32x16 sacc = {};
#pragma unroll
  for (int st = 0; st < 4; ++st) sacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[st], qf[st], sacc, 0, 0, 0);
  const float c2 = p.scale * 1.4426950408889634f;
  float m = -INFINITY;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int key = 8 * (j >> 2) + 4 * hi + (j & 3);
    sacc[j] = key < Z ? sacc[j] * c2 : -INFINITY;
    m = fmaxf(m, sacc[j]);
  }
  m = fmaxf(m, __shfl_xor(m, 32));
  float l = 0.f;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    sacc[j] = __builtin_amdgcn_exp2f(sacc[j] - m);  // masked keys: 2^-inf = 0
    l += sacc[j];
  }
  l += __shfl_xor(l, 32);

  // O^T = V^T P^T over two k-steps of 16 keys, two blocks of 32 dims.
  f32x16 oacc[2] = {};
#pragma unroll
  for (int kt = 0; kt < 2; ++kt) {
    bf16x8 pb;
#pragma unroll
    for (int mm = 0; mm < 8; ++mm) pb[mm] = (bf16)sacc[4 * (2 * kt + (mm >> 2)) + (mm & 3)];
#pragma unroll
    for (int db = 0; db < 2; ++db) {
      bf16x8 va;
#pragma unroll
      for (int mm = 0; mm < 8; ++mm) va[mm] = sw[at(16 * kt + 8 * (mm >> 2) + 4 * hi + (mm & 3), 32 * db + n)];
      oacc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, pb, oacc[db], 0, 0, 0);
    }
  }
  // The output goes back through the LDS buffer (row = query) so that each store
  // instruction writes whole 128-byte rows.
  const float inv = 1.f / l;
  wait_lgkm0();  // the V gathers are done
#pragma unroll
  for (int db = 0; db < 2; ++db)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const u32x2 ow = {pack_bf16x2(oacc[db][4 * i] * inv, oacc[db][4 * i + 1] * inv),
                        pack_bf16x2(oacc[db][4 * i + 2] * inv, oacc[db][4 * i + 3] * inv)};
      *(u32x2*)&sw[at(n, 32 * db + 8 * i + 4 * hi)] = ow;
    }
  wait_lgkm0();
  bf16* o = (bf16*)p.o + (int64_t)b * p.os[0] + (int64_t)y * p.os[2] + (int64_t)x * p.os[3] + (int64_t)h * p.os[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int r = lane / 8 + 8 * c;
    if (r < Z) *(u32x4*)(o + (int64_t)r * p.os[1] + 8 * (lane % 8)) = *(const u32x4*)&sw[at(r, 8 * (lane % 8))];
  }
  if (p.lse && hi == 0 && n < Z) p.lse[lse_index(p, b, n, y, x, h)] = m + __log2f(l);
#endif
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
template <typename T>
static int launch_scalar(const Na3dParams& p, hipStream_t st) {
  const int64_t total = (int64_t)p.B * p.H * p.ext[0] * p.ext[1] * p.ext[2];
  if (total == 0) return STRATA_HIP_OK;
  const int threads = 256;
  const int64_t blocks = (total + threads - 1) / threads;
  switch (p.D) {
#define STRATA_NA3D_SCALAR_CASE(DD)                                                            \
  case DD:                                                                                     \
    hipLaunchKernelGGL((na3d_scalar_kernel<T, DD>), dim3((unsigned)blocks), dim3(threads), 0, st, p, total); \
    break;
    STRATA_NA3D_SCALAR_CASE(8)
    STRATA_NA3D_SCALAR_CASE(16)
    STRATA_NA3D_SCALAR_CASE(32)
    STRATA_NA3D_SCALAR_CASE(64)
    STRATA_NA3D_SCALAR_CASE(128)
#undef STRATA_NA3D_SCALAR_CASE
    default:
      return fail(STRATA_HIP_EUNSUPPORTED, "na3d: head_dim must be one of 8, 16, 32, 64, 128");
  }
  return check_launch("na3d_scalar_kernel");
}

// fp32 tensors: the gather kernel on the matrix cores, else one thread per query.
static int launch_f32(const Na3dParams& p, hipStream_t st) {
  GatherParams g = {};
  g.c0 = p.q;
  g.s0 = p.k;
  g.s1 = p.v;
  g.o0 = p.o;
  g.B = p.B;
  g.H = p.H;
  g.D = p.D;
  for (int a = 0; a < 3; ++a) {
    g.L[a] = p.L[a];
    g.org[a] = p.org[a];
    g.ext[a] = p.ext[a];
    g.ker[a] = p.ker[a];
    g.dil[a] = p.dil[a];
  }
  for (int i = 0; i < 5; ++i) {
    g.cs[i] = p.qs[i];
    g.ss0[i] = p.ks[i];
    g.ss1[i] = p.vs[i];
    g.os[i] = p.os[i];
  }
  g.scale = p.scale;
  g.lse = p.lse;
  g.lse_ext1 = p.lse_ext1;
  return gather_plan(g, GATHER_FWD, 4) ? launch_gather(g, GATHER_FWD, false, st) : launch_scalar<float>(p, st);
}

// Query counts per axis of the box (largest over the dilation residue classes).
static void box_queries(const Na3dParams& p, int (&nq)[3]) {
  for (int a = 0; a < 3; ++a) {
    nq[a] = 0;
    for (int g = 0; g < p.dil[a]; ++g) {
      const int n = sub_end(p.org[a], p.ext[a], g, p.dil[a]) - sub_first(p.org[a], g, p.dil[a]);
      nq[a] = n > nq[a] ? n : nq[a];
    }
  }
}

// Workgroup tiles of the general kernel over the query box; false if the grid
// would not fit one launch.
template <int TX, int NTY>
static bool make_tiles(const Na3dParams& p, Na3dTiles& tg) {
  int nq[3];
  box_queries(p, nq);
  constexpr int TY = 16 / TX;
  tg.nzt = nq[0];
  tg.nyt = (nq[1] + NTY * TY - 1) / (NTY * TY);
  tg.nxt = (nq[2] + NA3D_NWX * TX - 1) / (NA3D_NWX * TX);
  tg.nres = p.dil[0] * p.dil[1] * p.dil[2];
  const int64_t total = (int64_t)tg.nxt * tg.nyt * tg.nzt * tg.nres * p.H * p.B;
  tg.total = total > 0x7fffffff ? 0 : (int)total;
  return total <= 0x7fffffff;
}

template <int D, int TX, int NTY, int RPS, int NBUF>
static int launch_mfma_cfg(const Na3dParams& p, hipStream_t st) {
  Na3dTiles tg;
  if (!make_tiles<TX, NTY>(p, tg)) return fail(STRATA_HIP_EUNSUPPORTED, "na3d: problem too large for one launch");
  const int total = tg.total;
  if (total == 0) return STRATA_HIP_OK;
  if (D >= 128)
    hipLaunchKernelGGL((na3d_mfma_wide_kernel<D, TX, NTY, RPS, NBUF>), dim3((unsigned)total), dim3(64 * NA3D_NWX), 0,
                       st, p, tg);
  else
    hipLaunchKernelGGL((na3d_mfma_kernel<D, TX, NTY, RPS, NBUF>), dim3((unsigned)total), dim3(64 * NA3D_NWX), 0, st, p,
                       tg);
  return check_launch("na3d_mfma_kernel");
}

// LDS budget per workgroup: ~80 KiB (two workgroups per CU).  A stage holds
// RPS key rows of K and of V.  Wide windows (4-column tiles, kx >= 10) take
// four rows per stage when a double-buffered ring of them fits the budget:
// half the stages, so half the per-stage barrier, DMA issue and LDS latency
// (configs[2]: 8.6 -> 8.2 ms).  Narrower windows keep two rows and a deeper
// ring: their shorter y-unions pad a 4-row stage and the ring would be 2 deep.
template <int D, int TX, int RPS>
constexpr int stage_bytes() {
  return 2 * RPS * (((NA3D_NWX - 1) * TX + 16 + 512 / D - 1) / (512 / D) * (512 / D)) * D * 2;
}
template <int D, int TX>
constexpr int rows_per_stage() {
  return TX <= 4 && 2 * stage_bytes<D, TX, 4>() <= 81920 ? 4 : 2;
}
// Ring depth: as deep as fits the budget, at most 4, at least double buffered.
constexpr int ring_depth(int stage_b) { return 81920 / stage_b >= 4 ? 4 : (81920 / stage_b >= 3 ? 3 : 2); }

template <int D, int TX, int NTY>
static int launch_mfma_tx(const Na3dParams& p, hipStream_t st) {
  constexpr int RPS = rows_per_stage<D, TX>();
  return launch_mfma_cfg<D, TX, NTY, RPS, ring_depth(stage_bytes<D, TX, RPS>())>(p, st);
}


// Strip kernel launch.  Work units are (batch, head, residue, z, column box)
// strips over the whole y range; the y range is cut into chunks only when the
// strips alone would not fill the GPU several times over.
// Strip work units over the query box; false if they would not fit one launch.
template <int TX>
static bool make_strips(const Na3dParams& p, Na3dStrips& sg) {
  constexpr int TY = 16 / TX;
  int nq[3];
  box_queries(p, nq);
  sg.nzt = nq[0];
  sg.nxt = (nq[2] + NA3D_NWX * TX - 1) / (NA3D_NWX * TX);
  sg.nres = p.dil[0] * p.dil[1] * p.dil[2];
  const int nty = (nq[1] + TY - 1) / TY;
  const int64_t strips = (int64_t)sg.nxt * sg.nzt * sg.nres * p.H * p.B;
  sg.nch = sg.cty = 1;
  sg.total = 0;
  if (strips == 0 || nty == 0) return true;
  int nch = 1;
  // Cut the y range into chunks only when the strips alone would leave the GPU
  // short of work: 4-column tiles aim at 2048 workgroups; the 2 x 8 tiles of
  // the small windows (one ramp of NS - 1 groups per chunk, short strips) at
  // one round of two workgroups per CU.
  const int target = TX == 8 ? 512 : 2048;
  while (strips * nch < target && nch < nty) ++nch;
  sg.cty = (nty + nch - 1) / nch;
  sg.nch = (nty + sg.cty - 1) / sg.cty;
  const int64_t total = strips * sg.nch;
  if (total > 0x7fffffff) return false;
  sg.total = (int)total;
  return true;
}

template <int D, int TX, int RPS, int NBUF, bool FAST, int KY = 13>
static int launch_strip(const Na3dParams& p, hipStream_t st) {
  Na3dStrips sg;
  if (!make_strips<TX>(p, sg)) return fail(STRATA_HIP_EUNSUPPORTED, "na3d: problem too large for one launch");
  const int total = sg.total;
  if (total == 0) return STRATA_HIP_OK;
  if constexpr (FAST) {
    if (p.lse)
      hipLaunchKernelGGL((na3d_strip_fast_kernel<D, TX, RPS, NBUF, KY, true>), dim3((unsigned)total),
                         dim3(64 * NA3D_NWX), 0, st, p, sg);
    else
      hipLaunchKernelGGL((na3d_strip_fast_kernel<D, TX, RPS, NBUF, KY, false>), dim3((unsigned)total),
                         dim3(64 * NA3D_NWX), 0, st, p, sg);
    return check_launch("na3d_strip_fast_kernel");
  } else {
    hipLaunchKernelGGL((na3d_strip_kernel<D, TX, RPS, NBUF>), dim3((unsigned)total), dim3(64 * NA3D_NWX), 0, st, p, sg);
    return check_launch("na3d_strip_kernel");
  }
}

// The strip kernel covers 4-column tiles (kx 10..13, ky <= 13) of head_dim 64
// with a window at least two slices deep (the next tile's Q is copied while the
// second slice of a group runs); its Q, K and V rows of one (batch, z, head)
// slice must fit 31-bit byte offsets (V may be a strided view of the qkv GEMM's
// output, three times the stride of a packed tensor).
static bool strip_fits(const Na3dParams& p) {
  if (p.D != 64 || p.ker[0] < 2 || p.ker[2] < 10 || p.ker[2] > 13) return false;
  // Taller windows keep more than four tiles alive per row group (the walk
  // would split into many short segments); row groups are packed in 10 bits.
  if (p.ker[1] > 13 || p.L[1] >= 4096) return false;
  const int64_t* sd[3] = {p.qs, p.ks, p.vs};
  for (int t = 0; t < 3; ++t)
    if (((int64_t)(p.L[1] - 1) * sd[t][2] + (int64_t)(p.L[2] - 1) * sd[t][3] + p.D) * 2 >= 0x7fffffffLL) return false;
  return true;
}

// Regular strips (na3d_strip_fast_kernel): ky = 13 and no query row of the box
// has a clamped y window in any residue class, so every tile's y-union starts
// one row group after the previous tile's.
static bool strip_regular(const Na3dParams& p) {
  if (p.ker[1] != 13) return false;
  const int r = p.ker[1] / 2, dy = p.dil[1];
  for (int g = 0; g < dy; ++g) {
    const int y0 = sub_first(p.org[1], g, dy), y1 = sub_end(p.org[1], p.ext[1], g, dy);
    if (y1 <= y0) continue;
    if (y0 - r < 0 || y1 - 1 + r > sub_len(p.L[1], g, dy) - 1) return false;
  }
  return true;
}

// Small windows on regular strips (na3d_strip_fast_kernel with 2 x 8 tiles and
// two rows per stage): head_dim 64, kx <= 9 (an 8-column tile's x-union fits one
// 16-key block), ky in {3, 5, 7, 9}, kz >= 2, no y dilation.
// Only query rows whose y window is not clamped form regular strips; the host
// splits the query box in y and gives the clamped edge rows to the general kernel.
static bool small_strip_fits(const Na3dParams& p) {
  if (p.D != 64 || p.ker[0] < 2 || p.ker[2] > 9 || p.dil[1] != 1) return false;
  if (p.ker[1] != 3 && p.ker[1] != 5 && p.ker[1] != 7 && p.ker[1] != 9) return false;
  if (p.L[1] >= 4096) return false;
  const int64_t* sd[3] = {p.qs, p.ks, p.vs};
  for (int t = 0; t < 3; ++t)
    if (((int64_t)(p.L[1] - 1) * sd[t][2] + (int64_t)(p.L[2] - 1) * sd[t][3] + p.D) * 2 >= 0x7fffffffLL) return false;
  return true;
}

template <int D>
static int launch_mfma_d(const Na3dParams& p, hipStream_t st);

// The query box restricted to rows [y0, y1) of itself (output pointer shifted).
static Na3dParams y_sub_box(const Na3dParams& p, int y0, int y1) {
  Na3dParams s = p;
  s.o = (char*)p.o + 2 * (int64_t)(y0 - p.org[1]) * p.os[2];
  if (p.lse) s.lse = p.lse + (int64_t)(y0 - p.org[1]) * p.ext[2] * p.H;
  s.org[1] = y0;
  s.ext[1] = y1 - y0;
  return s;
}

static int launch_small_strips(const Na3dParams& p, hipStream_t st) {
  const int kr = p.ker[1] / 2;
  const int y0 = p.org[1], y1 = p.org[1] + p.ext[1];
  const int r0 = y0 > kr ? y0 : kr, r1 = y1 < p.L[1] - kr ? y1 : p.L[1] - kr;
  if (r1 - r0 < 2) return launch_mfma_d<64>(p, st);
  // the clamped edge rows: at most kr = ky / 2 <= 4 at each end
  const Na3dParams mid = y_sub_box(p, r0, r1), e0 = y_sub_box(p, y0, r0), e1 = y_sub_box(p, r1, y1);
  Na3dStrips sg;
  Na3dTiles t0, t1;
  const bool ok = make_strips<8>(mid, sg) && (p.ker[1] <= 5 ? make_tiles<8, 1>(e0, t0) && make_tiles<8, 1>(e1, t1)
                                                            : make_tiles<8, 2>(e0, t0) && make_tiles<8, 2>(e1, t1));
  const int64_t n0 = (sg.total + 7) / 8 * 8, n1 = (t0.total + 7) / 8 * 8, total = n0 + n1 + t1.total;
  if (!ok || total > 0x7fffffff) return fail(STRATA_HIP_EUNSUPPORTED, "na3d: problem too large for one launch");
  if (total == 0) return STRATA_HIP_OK;
  const dim3 grid((unsigned)total), block(64 * NA3D_NWX);
  if (p.rc) {  // the queries' rotation in the kernel (inference: no lse)
    switch (p.ker[1]) {
      case 3:
        hipLaunchKernelGGL((na3d_small_fused_kernel<3, false, true>), grid, block, 0, st, mid, sg, e0, t0, e1, t1,
                           (int)n0, (int)n1);
        break;
      case 5:
        hipLaunchKernelGGL((na3d_small_fused_kernel<5, false, true>), grid, block, 0, st, mid, sg, e0, t0, e1, t1,
                           (int)n0, (int)n1);
        break;
      case 7:
        hipLaunchKernelGGL((na3d_small_fused_kernel<7, false, true>), grid, block, 0, st, mid, sg, e0, t0, e1, t1,
                           (int)n0, (int)n1);
        break;
      default:
        hipLaunchKernelGGL((na3d_small_fused_kernel<9, false, true>), grid, block, 0, st, mid, sg, e0, t0, e1, t1,
                           (int)n0, (int)n1);
        break;
    }
    return check_launch("na3d_small_fused_kernel (query RoPE)");
  }
  switch (p.ker[1]) {
    case 3:
      if (p.lse)
        hipLaunchKernelGGL((na3d_small_fused_kernel<3, true>), grid, block, 0, st, mid, sg, e0, t0, e1, t1, (int)n0,
                           (int)n1);
      else
        hipLaunchKernelGGL((na3d_small_fused_kernel<3, false>), grid, block, 0, st, mid, sg, e0, t0, e1, t1, (int)n0,
                           (int)n1);
      break;
    case 5:
      if (p.lse)
        hipLaunchKernelGGL((na3d_small_fused_kernel<5, true>), grid, block, 0, st, mid, sg, e0, t0, e1, t1, (int)n0,
                           (int)n1);
      else
        hipLaunchKernelGGL((na3d_small_fused_kernel<5, false>), grid, block, 0, st, mid, sg, e0, t0, e1, t1, (int)n0,
                           (int)n1);
      break;
    case 7:
      if (p.lse)
        hipLaunchKernelGGL((na3d_small_fused_kernel<7, true>), grid, block, 0, st, mid, sg, e0, t0, e1, t1, (int)n0,
                           (int)n1);
      else
        hipLaunchKernelGGL((na3d_small_fused_kernel<7, false>), grid, block, 0, st, mid, sg, e0, t0, e1, t1, (int)n0,
                           (int)n1);
      break;
    default:
      if (p.lse)
        hipLaunchKernelGGL((na3d_small_fused_kernel<9, true>), grid, block, 0, st, mid, sg, e0, t0, e1, t1, (int)n0,
                           (int)n1);
      else
        hipLaunchKernelGGL((na3d_small_fused_kernel<9, false>), grid, block, 0, st, mid, sg, e0, t0, e1, t1, (int)n0,
                           (int)n1);
      break;
  }
  return check_launch("na3d_small_fused_kernel");
}

template <int D>
static int launch_mfma_d(const Na3dParams& p, hipStream_t st) {
  constexpr int NTY = D >= 128 ? 2 : 4;
  const int kx = p.ker[2];
  if (kx == 1) return launch_mfma_tx<D, 16, NTY>(p, st);
  if (kx <= 9) return launch_mfma_tx<D, 8, NTY>(p, st);
  if (kx <= 13) return launch_mfma_tx<D, 4, NTY>(p, st);
  return launch_mfma_tx<D, 2, (NTY > 2 ? 2 : NTY)>(p, st);  // kx <= 15
}

static bool aligned16(const void* ptr) { return ((uintptr_t)ptr & 15u) == 0; }

// Depth-wise windows for na3d_column_kernel: (Z, 1, 1) with Z <= 32, undilated, head_dim
// 64, the whole grid as the query box (the MFMA layout conditions hold: na3d_mfma_ok).
static bool column_fits(const Na3dParams& p) {
  return p.D == 64 && p.ker[0] == p.L[0] && p.L[0] <= 32 && p.ker[1] == 1 && p.ker[2] == 1 && p.dil[0] == 1 &&
         p.dil[1] == 1 && p.dil[2] == 1 && p.org[0] == 0 && p.org[1] == 0 && p.org[2] == 0 && p.ext[0] == p.L[0] &&
         p.ext[1] == p.L[1] && p.ext[2] == p.L[2] && p.lse_ext1 == p.ext[1];
}

static int launch_column(const Na3dParams& p, hipStream_t st) {
  const int64_t items = (int64_t)p.B * p.L[1] * p.L[2] * p.H;
  const int64_t wgs = (items + 3) / 4;
  if (wgs > 0x7fffffff) return fail(STRATA_HIP_EUNSUPPORTED, "na3d: problem too large for one launch");
  hipLaunchKernelGGL(na3d_column_kernel, dim3((unsigned)wgs), dim3(256), 0, st, p, items);
  return check_launch("na3d_column_kernel");
}

// Query regions (na3d_region_kernel): kz = 3, ky in {3, 5, 7}, kx <= ky, head_dim 64;
// one slice of K and V rows must fit 31-bit byte offsets (as the strips).
// STRATA_HIP_NA3D_NO_REGIONS=1 switches the path off (the strips and the general
// kernel then take these windows; the tests compare the two).
static bool region_fits(const Na3dParams& p) {
  // Taken for ky = 3 only: at (3,3,3) it beats the small-window strips by ~18% (one
  // rollout tile: 1.21 -> 1.00 ms, with the query rotation 1.38 -> 1.14 ms); at (3,7,7)
  // over 8 query z's the strips stay ahead (the z ends' extra slot passes and each
  // workgroup's exposed first copies weigh more on an 8-slice walk than the saved
  // copies: configs[3] 0.363 against 0.333 ms).
  if (p.D != 64 || p.ker[0] != 3 || p.ker[1] != 3 || p.ker[2] > 3) return false;
  const int64_t* sd[2] = {p.ks, p.vs};
  for (int t = 0; t < 2; ++t)
    if (((int64_t)(p.L[1] - 1) * sd[t][2] + (int64_t)(p.L[2] - 1) * sd[t][3] + p.D) * 2 >= (int64_t)OOB) return false;
  // The z walk keeps at most four query z's live per stage s, the fourth being s - 2
  // or s + 2 (its slot is the one the interior leaves idle): every z sub-grid length
  // but 5 (where five overlap at s = 2).  Checked by brute force per residue class.
  for (int gz = 0; gz < p.dil[0]; ++gz) {
    const int Lz = sub_len(p.L[0], gz, p.dil[0]);
    const int z0 = sub_first(p.org[0], gz, p.dil[0]), z1 = sub_end(p.org[0], p.ext[0], gz, p.dil[0]);
    if (z1 <= z0) continue;
    for (int s = win_start(z0, Lz, 3); s < win_start(z1 - 1, Lz, 3) + 3; ++s) {
      int lo = 1 << 30, hi = -1, n = 0;
      for (int zq = z0; zq < z1; ++zq) {
        const int w = win_start(zq, Lz, 3);
        if (w <= s && s < w + 3) {
          lo = zq < lo ? zq : lo;
          hi = zq > hi ? zq : hi;
          ++n;
        }
      }
      if (n > 4 || hi - lo + 1 != n || lo < s - 2 || hi > s + 2 || (lo == s - 2 && hi == s + 2)) return false;
    }
  }
  return !std::getenv("STRATA_HIP_NA3D_NO_REGIONS");
}

template <int KY>
static int launch_region_ky(const Na3dParams& p, const Na3dRegions& rg, hipStream_t st) {
  const dim3 grid((unsigned)rg.total), block(512);
  if (p.rc)
    hipLaunchKernelGGL((na3d_region_kernel<KY, false, true>), grid, block, 0, st, p, rg);
  else if (p.lse)
    hipLaunchKernelGGL((na3d_region_kernel<KY, true, false>), grid, block, 0, st, p, rg);
  else
    hipLaunchKernelGGL((na3d_region_kernel<KY, false, false>), grid, block, 0, st, p, rg);
  return check_launch("na3d_region_kernel");
}

static int launch_region(const Na3dParams& p, hipStream_t st) {
  int nq[3];
  box_queries(p, nq);
  Na3dRegions rg;
  rg.nrx = (nq[2] + 15) / 16;
  rg.nry = (nq[1] + 7) / 8;
  rg.nres = p.dil[0] * p.dil[1] * p.dil[2];
  const int64_t total = (int64_t)rg.nrx * rg.nry * rg.nres * p.H * p.B;
  if (total > 0x7fffffff) return fail(STRATA_HIP_EUNSUPPORTED, "na3d: problem too large for one launch");
  rg.total = (int)total;
  if (total == 0 || nq[0] == 0) return STRATA_HIP_OK;
  return launch_region_ky<3>(p, rg, st);
}

}  // namespace strata

using namespace strata;

// Argument checks and kernel parameters shared by the forward entry points.
static int na3d_prepare(const strata_hip_na3d_args* a, Na3dParams& p) {
  if (!a) return fail(STRATA_HIP_EINVAL, "na3d: null args");
  if (!a->q || !a->k || !a->v || !a->out) return fail(STRATA_HIP_EINVAL, "na3d: null tensor pointer");
  if (a->dtype != STRATA_HIP_F32 && a->dtype != STRATA_HIP_BF16)
    return fail(STRATA_HIP_EINVAL, "na3d: dtype must be f32 or bf16");
  if (a->batch < 0 || a->heads <= 0 || a->head_dim <= 0) return fail(STRATA_HIP_EINVAL, "na3d: bad batch/heads/head_dim");
  static const char* axis = "zyx";
  for (int i = 0; i < 3; ++i) {
    const int L = a->grid[i], k = a->kernel[i], d = a->dilation[i];
    if (L <= 0) return fail(STRATA_HIP_EINVAL, std::string("na3d: grid size must be positive on axis ") + axis[i]);
    // Odd, or the whole undilated axis (every query then attends the full axis,
    // the window depth-wise attention uses along z).
    if (k <= 0 || ((k % 2) == 0 && !(k == L && d == 1)))
      return fail(STRATA_HIP_EINVAL,
                  std::string("na3d: kernel size must be odd and positive (or the whole axis) on axis ") + axis[i]);
    if (d <= 0) return fail(STRATA_HIP_EINVAL, std::string("na3d: dilation must be positive on axis ") + axis[i]);
    if ((int64_t)k * d > L)
      return fail(STRATA_HIP_EINVAL,
                  std::string("na3d: kernel_size * dilation exceeds the token grid on axis ") + axis[i]);
    if (a->q_origin[i] < 0 || a->q_extent[i] < 0 || a->q_origin[i] + a->q_extent[i] > L)
      return fail(STRATA_HIP_EINVAL, std::string("na3d: query box outside the grid on axis ") + axis[i]);
  }
  p.q = a->q;
  p.k = a->k;
  p.v = a->v;
  p.o = a->out;
  p.B = a->batch;
  p.H = a->heads;
  p.D = a->head_dim;
  for (int i = 0; i < 3; ++i) {
    p.L[i] = a->grid[i];
    p.org[i] = a->q_origin[i];
    p.ext[i] = a->q_extent[i];
    p.ker[i] = a->kernel[i];
    p.dil[i] = a->dilation[i];
  }
  for (int i = 0; i < 5; ++i) {
    p.qs[i] = a->q_stride[i];
    p.ks[i] = a->k_stride[i];
    p.vs[i] = a->v_stride[i];
    p.os[i] = a->o_stride[i];
  }
  p.scale = a->scale;
  p.lse = a->lse;
  p.lse_ext1 = a->q_extent[1];
  p.rc = p.rs = nullptr;
  p.rzt = 1;
  if (p.lse && ((uintptr_t)p.lse & 3u)) return fail(STRATA_HIP_EINVAL, "na3d: lse must be 4-byte aligned");
  return STRATA_HIP_OK;
}

// The bf16 MFMA kernels' layout conditions: 16-byte aligned tensors, strides in
// whole 16-byte chunks, and key/value rows that one buffer descriptor covers.
static bool na3d_mfma_ok(const Na3dParams& p) {
  bool mfma_ok = (p.D == 32 || p.D == 64 || p.D == 128) && p.ker[2] <= 15;
  if (mfma_ok) {
    const void* ptrs[4] = {p.q, p.k, p.v, p.o};
    const int64_t* strides[4] = {p.qs, p.ks, p.vs, p.os};
    for (int t = 0; t < 4; ++t) {
      if (!aligned16(ptrs[t])) mfma_ok = false;
      for (int i = 0; i < 5; ++i)
        if (strides[t][i] % 8 != 0) mfma_ok = false;
    }
  }
  if (mfma_ok) {
    // One buffer descriptor covers a pair of (z, y) key rows with 31-bit byte
    // offsets: the x extent of a row must fit inside the row stride, two row
    // strides must stay below the out-of-range offset, strides must be
    // positive, and a workgroup's y-union (<= 16 + ky - 1 rows) must fit the
    // 32-bit per-pair masks.
    const int64_t* kv[2] = {p.ks, p.vs};
    for (int t = 0; t < 2; ++t) {
      const int64_t* sd = kv[t];
      for (int i = 0; i < 5; ++i)
        if (sd[i] <= 0 && !(i == 0 && p.B == 1) && !(i == 4 && p.H == 1)) mfma_ok = false;
      if ((int64_t)(p.L[2] - 1) * sd[3] + p.D > sd[2]) mfma_ok = false;
      if (4 * (int64_t)p.dil[1] * sd[2] * 2 >= (int64_t)OOB) mfma_ok = false;
    }
    if (16 + p.ker[1] - 1 > 64) mfma_ok = false;
  }
  return mfma_ok;
}

extern "C" int strata_hip_na3d_fwd(const strata_hip_na3d_args* a, void* stream) {
  Na3dParams p;
  if (const int rc = na3d_prepare(a, p)) return rc;
  if ((int64_t)p.B * p.ext[0] * p.ext[1] * p.ext[2] == 0) return STRATA_HIP_OK;
  hipStream_t st = (hipStream_t)stream;
  if (a->dtype == STRATA_HIP_F32) return launch_f32(p, st);
  const bool mfma_ok = na3d_mfma_ok(p);
  if (!mfma_ok) return launch_scalar<bf16>(p, st);
  if (column_fits(p)) return launch_column(p, st);
  switch (p.D) {
    case 32:
      return launch_mfma_d<32>(p, st);
    case 64:
      if (region_fits(p)) return launch_region(p, st);
      if (strip_fits(p))
        return strip_regular(p) ? launch_strip<64, 4, 4, 2, true>(p, st) : launch_strip<64, 4, 4, 2, false>(p, st);
      if (small_strip_fits(p) && !std::getenv("STRATA_HIP_NA3D_NO_SMALL_STRIPS")) return launch_small_strips(p, st);
      return launch_mfma_d<64>(p, st);
    default:
      return launch_mfma_d<128>(p, st);
  }
}

// The query-RoPE forward's checks; fills p with the tables set.
static int rope_q_setup(const strata_hip_na3d_args* a, const float* cos, const float* sin, int32_t table_z,
                        Na3dParams& p) {
  if (const int rc = na3d_prepare(a, p)) return rc;
  if (!cos || !sin) return fail(STRATA_HIP_EINVAL, "na3d_fwd_rope_q: null cos or sin table");
  if (((uintptr_t)cos & 15u) || ((uintptr_t)sin & 15u))
    return fail(STRATA_HIP_EINVAL, "na3d_fwd_rope_q: cos and sin must be 16-byte aligned");
  if (table_z != 1 && table_z != p.L[0]) return fail(STRATA_HIP_EINVAL, "na3d_fwd_rope_q: table_z must be 1 or the grid's z");
  if (a->dtype != STRATA_HIP_BF16 || p.D != 64 || p.lse)
    return fail(STRATA_HIP_EUNSUPPORTED, "na3d_fwd_rope_q: bf16, head_dim 64 and no lse output only");
  for (int i = 0; i < 3; ++i)
    if (p.org[i] != 0 || p.ext[i] != p.L[i])
      return fail(STRATA_HIP_EUNSUPPORTED, "na3d_fwd_rope_q: the query box must be the full grid");
  if ((int64_t)p.B * table_z * p.L[1] * p.L[2] * 128 >= (int64_t)OOB)
    return fail(STRATA_HIP_EUNSUPPORTED, "na3d_fwd_rope_q: tables too large for 31-bit offsets");
  const int kr = p.ker[1] / 2;
  const int r0 = p.org[1] > kr ? p.org[1] : kr, r1 = p.org[1] + p.ext[1] < p.L[1] - kr ? p.org[1] + p.ext[1] : p.L[1] - kr;
  const bool mfma_ok = na3d_mfma_ok(p);
  if (!(mfma_ok && region_fits(p)) && (!mfma_ok || strip_fits(p) || !small_strip_fits(p) || r1 - r0 < 2 ||
                                       std::getenv("STRATA_HIP_NA3D_NO_SMALL_STRIPS")))
    return fail(STRATA_HIP_EUNSUPPORTED,
                "na3d_fwd_rope_q: this window or layout runs a kernel without the query rotation "
                "(rotate q in strata_hip_rope_qkv_pack and call strata_hip_na3d_fwd)");
  p.rc = cos;
  p.rs = sin;
  p.rzt = table_z;
  return STRATA_HIP_OK;
}

extern "C" int strata_hip_na3d_fwd_rope_q_supported(const strata_hip_na3d_args* a, const float* cos, const float* sin,
                                                    int32_t table_z) {
  Na3dParams p;
  return rope_q_setup(a, cos, sin, table_z, p) == STRATA_HIP_OK ? 1 : 0;
}

extern "C" int strata_hip_na3d_fwd_rope_q(const strata_hip_na3d_args* a, const float* cos, const float* sin,
                                          int32_t table_z, void* stream) {
  Na3dParams p;
  if (const int rc = rope_q_setup(a, cos, sin, table_z, p)) return rc;
  if ((int64_t)p.B * p.ext[0] * p.ext[1] * p.ext[2] == 0) return STRATA_HIP_OK;
  // the region or the small-window launch (rope_q_setup checked that one applies)
  return region_fits(p) ? launch_region(p, (hipStream_t)stream) : launch_small_strips(p, (hipStream_t)stream);
}
