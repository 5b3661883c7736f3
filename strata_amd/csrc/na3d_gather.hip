// NA3D forward and backward in fp32 arithmetic on v_mfma_f32_16x16x4_f32.
//
// A wave owns a tile of 16 column tokens and walks the union of their windows 16
// row tokens at a time, straight from global memory: no LDS staging, no shuffles
// between the two products.  With columns on the MFMA's N and rows on its M,
//   S = rows x columns:  A = the rows' dims, B = the columns' dims.  The order of
//       the contraction is free as long as both sides agree, so lane (n, g)
//       = (lane & 15, lane >> 4) takes dims 16i + 4g + e: 16-byte loads, four
//       lanes on 64 contiguous bytes of a token.
//   O^T += R^T W:  A = the rows transposed (lane: dims CW (n + 16j) + e of row
//       4g + s, whole tokens per load), B = the weights.  A lane's accumulator of
//       S holds rows 4g + s of column n, exactly the B operand of step s.
// The forward's weights are the softmax probabilities (online, per column), the
// backward's dS (and P): dq streams k and v under 16 queries, dk / dv stream q and
// dO under 16 keys (their inverse windows are boxes too).  Rows outside a column's
// window carry weight 0; a non-finite row value would still turn 0 x inf into NaN
// there, so such a block of rows (one check per block) is added on the VALU for
// the columns whose window holds it.
//
// bf16 tensors (the backward): S and dP are bf16 products, exact in the fp32
// accumulator, so they run on the 16 x faster v_mfma_f32_16x16x32_bf16 (the scale
// applied to the scores instead of the columns); the fp32 weights enter the second
// product as two bf16 terms, w = hi + lo to 2^-17, two v_mfma_f32_16x16x16_bf16
// in the place of four fp32 steps.  The gradients' error against float64, over the
// VALU kernels' with fp32 weights, at 24 drawn shapes (head_dim 32, 64, 128, dilation
// 1, 2): 0.9998 .. 1.0003, mean 1.0000 (the bf16 outputs round 2^8 times coarser).
// A weight that bf16 does not hold (infinite, NaN) takes the VALU branch in fp32.
//
// The union is a box per tile; its rows' offsets and coordinates go through a
// table in LDS (512 rows at a time, built by the wave), which makes any window,
// dilation and stride alike.  The tile's shape (16 = tz x ty x tx) is the one with
// the fewest row blocks: 4 x 4 in y, x for square windows, 16 along z for (Z, 1, 1).
//
// fp32 is bound by issue: at (3,7,7), head_dim 64 the matrix cores are busy for 46-50%
// of the time (1024 cycles per 16 x 16 block forward, 49% of whose pairs are useful)
// and the VALU for 28-52%, waves wait 13-17%.  bf16: VALU 56-58%, matrix cores 12-14%,
// waves wait for the rows 32-42%.
// Few tiles: SPLIT waves share one tile's rows and merge in LDS.  Measured, us,
// a thread (backward: four lanes) per token -> here:
//   fp32 forward  [1,4,16,16,4,32] (3,5,5)      134 -> 8.9
//   fp32 backward [1,16,64,64,8,64] (3,7,7)    7650 -> 1850 (forward 525, 37 TFLOP/s)
//                 [1,8,64,64,8,128] (3,7,7)   12930 -> 1950 .. 2140
//   bf16 backward [1,16,64,64,8,64] (3,7,7) dilation 2   2190 -> 900
//                 [1,8,40,52,8,32] (3,9,9)      877 -> 210
//                 [1,16,64,64,8,64] (3,3,3) dilation 2    519 -> 436
#include <cstdlib>
#include <type_traits>

#include "na3d_gather.h"

namespace strata {

constexpr int GATHER_ROWS = 512;  // row tokens per table

// 0x7f80 or more in either half: that bf16 is infinite or NaN.
__device__ __forceinline__ uint32_t gather_max_exp(uint32_t a, uint32_t w) {
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a),
                                                                __builtin_bit_cast(u16x2, w & 0x7fff7fffu)));
}

// CW consecutive values (4, or 2 at head_dim 32): fp32 in the first CW of a quad,
// bf16 as pairs.
template <typename T, int CW>
__device__ __forceinline__ auto gather_ldc(const T* p) {
  if constexpr (sizeof(T) == 4) {
    if constexpr (CW == 4) return *(const f32x4*)p;
    else return (f32x4){p[0], p[1], 0.f, 0.f};
  } else {
    if constexpr (CW == 4) return *(const u32x2*)p;
    else return (u32x2){*(const uint32_t*)p, 0u};
  }
}

template <typename T, int D, int MODE, int SPLIT>
__global__ __launch_bounds__(256) void na3d_gather_kernel(GatherParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int CW = D >= 64 ? 4 : 2;        // consecutive dims per lane in the transposed loads
  constexpr int NJ = D / (16 * CW);          // such runs per lane
  constexpr int NB = NJ * CW;                // accumulator blocks of 16 dims
  constexpr bool BWD = MODE != GATHER_FWD;
  constexpr int NACC = MODE == GATHER_DKV ? 2 : 1;
  constexpr float LOG2E = 1.4426950408889634f;
  constexpr bool HALF = sizeof(T) == 2;
  constexpr int NR = HALF ? D / 32 : D / 16;     // MFMA operand runs of a token (8 bf16 or 4 fp32 each)
  typedef typename std::conditional<HALF, bf16x8, f32x4>::type Run;
  typedef typename std::conditional<HALF, u32x2, f32x4>::type Quad;  // CW values of a token
  constexpr int RUN = HALF ? 32 : 16, RLANE = HALF ? 8 : 4;
  constexpr int MERGE = SPLIT > 1 ? (SPLIT - 1) * (4 / SPLIT) * 64 * (NACC * NB * 4 + 2) : 1;  // floats
  constexpr int TABLE = 4 * GATHER_ROWS * 3;
  __shared__ __attribute__((aligned(16))) int lds[MERGE > TABLE ? MERGE : TABLE];

  const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int part = wave % SPLIT;
  int tile = xcd_tile_order((int)gridDim.x, (int)__builtin_amdgcn_workgroup_id_x()) * (4 / SPLIT) + wave / SPLIT;
  bool live = tile < p.tiles;  // uniform per wave; an idle wave still meets the merge barriers
  if (!live) tile = 0;

  int w = tile;
  int tc[3];
  for (int a = 2; a >= 0; --a) {
    tc[a] = w % p.nt[a];
    w /= p.nt[a];
  }
  int res = w % p.nres;
  w /= p.nres;
  const int h = w % p.H, b = w / p.H;
  int rg[3];  // dilation residue per axis
  for (int a = 2; a >= 0; --a) {
    rg[a] = res % p.dil[a];
    res /= p.dil[a];
  }

  // Per axis (sub-grid coordinates): the lane's column token, its window
  // [lo, lo + cnt) relative to the union's origin u0, and the union's extent.
  int u0[3], U[3], lo[3], cnt[3], cc[3];
  bool valid = true;
  {
    int li = n;
    for (int a = 2; a >= 0; --a) {
      const int d = p.dil[a], k = p.ker[a], Lg = sub_len(p.L[a], rg[a], d);
      const int q1 = sub_end(p.org[a], p.ext[a], rg[a], d);
      const int q0 = sub_first(p.org[a], rg[a], d) + (tc[a] << p.tl[a]);
      const int t = li & ((1 << p.tl[a]) - 1);
      li >>= p.tl[a];
      if (q0 >= q1) live = false;
      valid = valid && q0 + t < q1;
      auto win = [&](int j, int& first, int& count) {
        if constexpr (MODE == GATHER_DKV) {  // the queries whose windows hold key j
          const int r = k / 2;
          first = j - k + 1 <= 0 ? 0 : j - k + 1 + r;
          count = (j >= Lg - k ? Lg - 1 : j + r) - first + 1;
        } else {
          first = win_start(j, Lg, k);
          count = k;
        }
      };
      int f, c;
      win(min(q0, max(q1 - 1, 0)), f, c);
      u0[a] = f;
      win(max(min(q0 + (1 << p.tl[a]) - 1, q1 - 1), 0), f, c);
      U[a] = f + c - u0[a];
      const int j = max(min(q0 + t, q1 - 1), 0);
      win(j, f, c);
      lo[a] = f - u0[a];
      cnt[a] = c;
      cc[a] = rg[a] + d * j;  // full-grid coordinate
    }
  }
  const int64_t coff = b * p.cs[0] + cc[0] * p.cs[1] + cc[1] * p.cs[2] + cc[2] * p.cs[3] + h * p.cs[4];
  const int64_t cidx = (((int64_t)b * p.L[0] + cc[0]) * p.L[1] + cc[1]) * (int64_t)p.L[2] * p.H + (int64_t)cc[2] * p.H + h;
  int64_t sb0 = b * p.ss0[0] + h * p.ss0[4], sb1 = b * p.ss1[0] + h * p.ss1[4];
  int st0[3], st1[3];
  for (int a = 0; a < 3; ++a) {
    const int64_t c0 = rg[a] + (int64_t)p.dil[a] * u0[a];
    sb0 += c0 * p.ss0[1 + a];
    sb1 += c0 * p.ss1[1 + a];
    st0[a] = (int)(p.dil[a] * p.ss0[1 + a]);
    st1[a] = (int)(p.dil[a] * p.ss1[1 + a]);
  }
  const T* s0 = (const T*)p.s0 + sb0;
  const T* s1 = (const T*)p.s1 + sb1;
  // the backward's tensors are contiguous: statistics at (element offset) / D
  const float* lse_s = BWD ? p.lse + sb0 / D : nullptr;
  const float* dsum_s = BWD ? p.dsum + sb0 / D : nullptr;

  // The columns' operand(s); the backward's scores are in log2 units.
  Run ca[NR], cb[BWD ? NR : 1];
  const float c2 = BWD ? p.scale * LOG2E : p.scale;
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    ca[i] = *(const Run*)((const T*)p.c0 + coff + RUN * i + RLANE * g);
    if constexpr (!HALF) ca[i] *= c2;
    if constexpr (BWD) cb[i] = *(const Run*)((const T*)p.c1 + coff + RUN * i + RLANE * g);
  }
  float lse_c = 0.f, dsum_c = 0.f;
  if constexpr (MODE == GATHER_DQ) {
    lse_c = p.lse[cidx];
    dsum_c = p.dsum[cidx];
  }

  f32x4 acc[NACC][NB];
#pragma unroll
  for (int x = 0; x < NACC; ++x)
#pragma unroll
    for (int i = 0; i < NB; ++i) acc[x][i] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  int* t0 = lds + wave * GATHER_ROWS * 3;
  int* t1 = t0 + GATHER_ROWS;
  int* tx = t1 + GATHER_ROWS;
  const int total = live ? U[0] * U[1] * U[2] : 0;
  const int nblk = (total + 15) / 16;
  const int blk0 = nblk * part / SPLIT, blk1 = nblk * (part + 1) / SPLIT;

  for (int base = blk0; base < blk1; base += GATHER_ROWS / 16) {
    const int nb = min(GATHER_ROWS / 16, blk1 - base);
    // table of this chunk's rows (wave-private; the last block's reads are done)
    wait_lgkm0();
    for (int i = lane; i < nb * 16; i += 64) {
      const int f = base * 16 + i;
      int zr = 0, yr = 0, xr = 0;
      if (f < total) {
        xr = f % U[2];
        const int r = f / U[2];
        yr = r % U[1];
        zr = r / U[1];
      }
      t0[i] = zr * st0[0] + yr * st0[1] + xr * st0[2];
      t1[i] = zr * st1[0] + yr * st1[1] + xr * st1[2];
      tx[i] = zr | yr << 10 | xr << 20;
    }
    wait_lgkm0();
    __builtin_amdgcn_wave_barrier();

    auto load_rows = [&](const T* s, const int* t, int blk, Run (&r)[NR]) {
      const T* q = s + t[blk * 16 + n] + RLANE * g;
#pragma unroll
      for (int i = 0; i < NR; ++i) r[i] = *(const Run*)(q + RUN * i);
    };
    auto load_trans = [&](const T* s, const int (&off)[4], Quad (&r)[4][NJ]) {
#pragma unroll
      for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int j = 0; j < NJ; ++j) r[st][j] = gather_ldc<T, CW>(s + off[st] + CW * (n + 16 * j));
    };
    auto product = [&](const Run (&r)[NR], const Run (&c)[NR]) {
      if constexpr (HALF) {
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < NR; ++i) s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(r[i], c[i], s, 0, 0, 0);
        return s;
      } else {
        // four partial sums: a chain over all D dims rounds D / 4 times in a row
        // (the gradients' error against float64 1.3 x that of this form)
        f32x4 s[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s[e] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int i = 0; i < NR; ++i) s[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(r[i][e], c[i][e], s[e], 0, 0, 0);
        }
        return (s[0] + s[1]) + (s[2] + s[3]);
      }
    };
    // acc += rows^T x weights; in: bit r = row 4g + r lies in the column's window
    auto accumulate = [&](f32x4 (&o)[NB], const Quad (&r)[4][NJ], const float (&wt)[4], const T* s, const int* t,
                          int blk, int in) {
      bool bad;  // some row value is not finite, or (two terms of it: inf - inf) some bf16 weight
      u32x2 hi = {0u, 0u};
      if constexpr (HALF) {
        hi = (u32x2){pack_bf16x2(wt[0], wt[1]), pack_bf16x2(wt[2], wt[3])};
        uint32_t x = gather_max_exp(gather_max_exp(0, hi[0]), hi[1]);
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
          for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int e = 0; e < CW / 2; ++e) x = gather_max_exp(x, r[st][j][e]);
        bad = (x & 0xffffu) >= 0x7f80u || (x >> 16) >= 0x7f80u;
      } else {
        float z = 0.f;
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
          for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int e = 0; e < CW; ++e) z = fmaf(r[st][j][e], 0.f, z);
        bad = z != 0.f;
      }
      if (__builtin_expect(__any(bad), 0)) {
        for (int row = 0; row < 16; ++row) {
          const int src = (row >> 2) * 16 + n;
          float wv = 0.f;
#pragma unroll
          for (int st = 0; st < 4; ++st) {
            const float v = __shfl(wt[st], src);
            if (st == (row & 3)) wv = v;
          }
          const int inw = __shfl(in, src);
          if (inw >> (row & 3) & 1) {
            const T* q = s + t[blk * 16 + row];
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
              for (int e = 0; e < CW; ++e)
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4)
                  o[j * CW + e][r4] = fmaf(wv, (float)q[CW * (4 * g + r4 + 16 * j) + e], o[j * CW + e][r4]);
          }
        }
        return;
      }
      if constexpr (HALF) {
        typedef short s16x4 __attribute__((ext_vector_type(4)));
        const u32x2 lw = {pack_bf16x2(wt[0] - bf16_lo(hi[0]), wt[1] - bf16_hi(hi[0])),
                          pack_bf16x2(wt[2] - bf16_lo(hi[1]), wt[3] - bf16_hi(hi[1]))};
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int e = 0; e < CW; ++e) {
            // dim e of rows 4g .. 4g + 3: halves of four dwords
            const uint32_t sel = e & 1 ? 0x07060302u : 0x05040100u;
            const u32x2 a = {__builtin_amdgcn_perm(r[1][j][e / 2], r[0][j][e / 2], sel),
                             __builtin_amdgcn_perm(r[3][j][e / 2], r[2][j][e / 2], sel)};
            f32x4& x = o[j * CW + e];
            x = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, lw),
                                                          x, 0, 0, 0);
            x = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, hi),
                                                          x, 0, 0, 0);
          }
      } else {
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
          for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int e = 0; e < CW; ++e)
              o[j * CW + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(r[st][j][e], wt[st], o[j * CW + e], 0, 0, 0);
      }
    };

    Run ra[NR];
    load_rows(s0, t0, 0, ra);
    for (int blk = 0; blk < nb; ++blk) {
      int off0[4], off1[4], crd[4], in = 0;
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        off0[st] = t0[blk * 16 + 4 * g + st];
        off1[st] = t1[blk * 16 + 4 * g + st];
        crd[st] = tx[blk * 16 + 4 * g + st];
      }
      // this block's remaining operands, then the next block's first one
      Run rb[BWD ? NR : 1];
      Quad rt0[BWD ? 4 : 1][NJ], rt1[4][NJ];
      float ls[4], ds[4];
      if constexpr (BWD) load_rows(s1, t1, blk, rb);
      if constexpr (MODE == GATHER_FWD || MODE == GATHER_DKV) load_trans(s1, off1, rt1);
      if constexpr (BWD) load_trans(s0, off0, rt0);
      if constexpr (MODE == GATHER_DKV) {
#pragma unroll
        for (int st = 0; st < 4; ++st) {
          ls[st] = lse_s[off0[st] / D];
          ds[st] = dsum_s[off0[st] / D];
        }
      }
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        const int zr = crd[st] & 1023, yr = crd[st] >> 10 & 1023, xr = crd[st] >> 20;
        const bool ok = (base + blk) * 16 + 4 * g + st < total && (unsigned)(zr - lo[0]) < (unsigned)cnt[0] &&
                        (unsigned)(yr - lo[1]) < (unsigned)cnt[1] && (unsigned)(xr - lo[2]) < (unsigned)cnt[2];
        in |= (int)ok << st;
      }
      f32x4 s = product(ra, ca);
      load_rows(s0, t0, min(blk + 1, nb - 1), ra);
      float wt[4];
      if constexpr (MODE == GATHER_FWD) {
        float bm = -INFINITY;
#pragma unroll
        for (int st = 0; st < 4; ++st)
          if (in >> st & 1) bm = fmaxf(bm, s[st]);
        bm = fmaxf(bm, __shfl_xor(bm, 16));
        bm = fmaxf(bm, __shfl_xor(bm, 32));
        const float mn = fmaxf(m, bm);
        // no finite score yet: keep the reference at 0 (exp(-inf - 0) = 0)
        const float ref = mn == -INFINITY ? 0.f : mn;
        if (__any(mn != m)) {
          const float alpha = expf(m - ref);
          l *= alpha;
#pragma unroll
          for (int i = 0; i < NB; ++i) acc[0][i] *= alpha;
        }
        m = mn;
#pragma unroll
        for (int st = 0; st < 4; ++st) {
          wt[st] = in >> st & 1 ? expf(s[st] - ref) : 0.f;
          l += wt[st];
        }
        accumulate(acc[0], rt1, wt, s1, t1, blk, in);
      } else {
        const f32x4 dp = product(rb, cb);
        float pr[4];
#pragma unroll
        for (int st = 0; st < 4; ++st) {
          const bool ok = in >> st & 1;
          const float lv = MODE == GATHER_DQ ? lse_c : ls[st], dv = MODE == GATHER_DQ ? dsum_c : ds[st];
          pr[st] = ok ? exp2f((HALF ? s[st] * c2 : s[st]) - lv) : 0.f;
          wt[st] = ok ? pr[st] * (dp[st] - dv) : 0.f;
        }
        accumulate(acc[0], rt0, wt, s0, t0, blk, in);
        if constexpr (MODE == GATHER_DKV) accumulate(acc[1], rt1, pr, s1, t1, blk, in);
      }
    }
  }

  if constexpr (MODE == GATHER_FWD) {
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
  }
  if constexpr (SPLIT > 1) {  // the parts of a tile, merged into part 0 in part order
    constexpr int REC = NACC * NB * 4 + 2;
    __syncthreads();  // every wave is done with its table
    float* f = (float*)lds;
    if (part > 0) {
      float* r = f + (((wave / SPLIT) * (SPLIT - 1) + part - 1) * REC) * 64 + lane;
#pragma unroll
      for (int x = 0; x < NACC; ++x)
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) r[((x * NB + i) * 4 + e) * 64] = acc[x][i][e];
      r[(REC - 2) * 64] = m;
      r[(REC - 1) * 64] = l;
    }
    __syncthreads();
    if (part > 0) return;
    for (int q = 0; q < SPLIT - 1; ++q) {
      const float* r = f + (((wave / SPLIT) * (SPLIT - 1) + q) * REC) * 64 + lane;
      float fa = 1.f, fb = 1.f;
      if constexpr (MODE == GATHER_FWD) {
        const float mq = r[(REC - 2) * 64], mn = fmaxf(m, mq), ref = mn == -INFINITY ? 0.f : mn;
        fa = expf(m - ref);
        fb = expf(mq - ref);
        l = l * fa + r[(REC - 1) * 64] * fb;
        m = mn;
      }
#pragma unroll
      for (int x = 0; x < NACC; ++x)
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[x][i][e] = acc[x][i][e] * fa + r[((x * NB + i) * 4 + e) * 64] * fb;
    }
  }
  if (!live || !valid) return;

  // Block (j, e) row 4g + r is dim CW (4g + r + 16j) + e: 4 CW contiguous dims per j.
  int64_t oo = b * p.os[0] + h * p.os[4];
  for (int a = 0; a < 3; ++a) oo += (int64_t)(cc[a] - p.org[a]) * p.os[1 + a];
  const float m0 = MODE == GATHER_FWD ? 1.f / l : p.scale;
#pragma unroll
  for (int x = 0; x < NACC; ++x) {
    T* o = (T*)(x == 0 ? p.o0 : p.o1) + oo;
    const float mul = x == 0 ? m0 : 1.f;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      float v[4 * CW];
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int e = 0; e < CW; ++e) v[CW * r + e] = acc[x][j * CW + e][r] * mul;
      T* q = o + CW * 4 * g + 16 * CW * j;
#pragma unroll
      for (int i = 0; i < CW; ++i) {
        if constexpr (sizeof(T) == 4) {
          *(f32x4*)(q + 4 * i) = (f32x4){v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
        } else {
          *(u32x2*)(q + 4 * i) = (u32x2){pack_bf16x2(v[4 * i], v[4 * i + 1]), pack_bf16x2(v[4 * i + 2], v[4 * i + 3])};
        }
      }
    }
  }
  if constexpr (MODE == GATHER_FWD) {
    if (p.lse && g == 0)
      p.lse[((((int64_t)b * p.ext[0] + cc[0] - p.org[0]) * p.lse_ext1 + cc[1] - p.org[1]) * p.ext[2] + cc[2] -
             p.org[2]) * p.H + h] = (m + logf(l)) * LOG2E;
  }
#endif
}

// Most rows the union of a tile of t columns holds along axis a.  A window is k rows and
// moves with its query: k + t - 1.  An inverse window is k rows in the interior and k / 2 more
// where one end of the axis clamps; on an axis so short that one tile holds a key clamped at
// the start (j < k) and one clamped at the end (j >= n - k), the union is the axis.
static int64_t union_max(const GatherParams& p, int a, int t, int mode) {
  const int64_t k = p.ker[a], d = p.dil[a];
  auto rows = [&](int64_t n) -> int64_t {  // n: the length of a residue class
    if (mode != GATHER_DKV) return n < k + t - 1 ? n : k + t - 1;
    return n <= 2 * k + t - 2 ? n : k + k / 2 + t - 1;
  };
  const int64_t u0 = rows((p.L[a] + d - 1) / d), u1 = rows(p.L[a] / d);
  return u0 > u1 ? u0 : u1;
}

bool gather_plan(GatherParams& p, int mode, int elem_bytes) {
  if (p.D != 32 && p.D != 64 && p.D != 128) return false;
  const int align = 16 / elem_bytes;  // every load and store of a token moves at most 16 bytes
  const void* ptrs[6] = {p.c0, p.c1 ? p.c1 : p.c0, p.s0, p.s1, p.o0, p.o1 ? p.o1 : p.o0};
  for (const void* q : ptrs)
    if ((uintptr_t)q & 15u) return false;
  const int64_t* strides[4] = {p.cs, p.ss0, p.ss1, p.os};
  for (const int64_t* s : strides)
    for (int i = 0; i < 5; ++i)
      if (s[i] % align) return false;
  int nq[3];
  for (int a = 0; a < 3; ++a) {
    nq[a] = 0;
    for (int r = 0; r < p.dil[a]; ++r) {
      const int c = sub_end(p.org[a], p.ext[a], r, p.dil[a]) - sub_first(p.org[a], r, p.dil[a]);
      nq[a] = c > nq[a] ? c : nq[a];
    }
  }
  p.nres = p.dil[0] * p.dil[1] * p.dil[2];
  // The tile shape with the fewest row blocks over all tiles, of those whose union the row
  // table describes: 10-bit coordinates, 32-bit element offsets.
  int64_t best = INT64_MAX;
  for (int lz = 0; lz <= 4; ++lz)
    for (int ly = 0; ly + lz <= 4; ++ly) {
      const int lg[3] = {lz, ly, 4 - lz - ly};
      int64_t tiles = 1, rows = 1, span0 = p.D, span1 = p.D;
      bool fits = true;
      for (int a = 0; a < 3; ++a) {
        const int64_t u = union_max(p, a, 1 << lg[a], mode);
        const int64_t d0 = std::abs(p.ss0[1 + a] * p.dil[a]), d1 = std::abs(p.ss1[1 + a] * p.dil[a]);
        tiles *= (nq[a] + (1 << lg[a]) - 1) >> lg[a];
        rows *= u;
        fits = u <= 1024 && d0 <= 0x7fffffff && d1 <= 0x7fffffff;
        if (!fits) break;
        span0 += (u - 1) * d0;
        span1 += (u - 1) * d1;
      }
      if (!fits || span0 > 0x7fffffff || span1 > 0x7fffffff) continue;
      const int64_t cost = tiles * ((rows + 15) / 16);
      if (cost < best) {
        best = cost;
        for (int a = 0; a < 3; ++a) p.tl[a] = lg[a];
      }
    }
  if (best == INT64_MAX) return false;
  int64_t tiles = (int64_t)p.B * p.H * p.nres;
  for (int a = 0; a < 3; ++a) {
    p.nt[a] = (nq[a] + (1 << p.tl[a]) - 1) >> p.tl[a];
    tiles *= p.nt[a];
  }
  p.tiles = (int)tiles;
  return tiles <= 0x7ffffff0;
}

// Waves that share one tile's rows.  8 waves per CU hide the loads (two per SIMD); a problem with
// fewer tiles splits each over 2 or 4.  The parts' sums are merged, so the split shows in the last
// bits: it goes by the tiles of one sample, and a sample's result does not depend on its batch.
// That costs batches of small samples up to a fifth against the split for the whole call: us at
// 1 / 4 / 16 samples of [4,16,16,4,32] (3,5,5), 256 tiles, fp32 backward 31 / 42 / 110 (whole
// call 31 / 38 / 101); of [8,24,24,4,128] (3,5,5), 1152 tiles, forward 47 / 142 / 562 (47 / 129 / 482).
int gather_split(const GatherParams& p) {
  constexpr int WANT = 2048;
  const int tiles = p.tiles / p.B;
  return tiles >= WANT ? 1 : tiles >= WANT / 2 ? 2 : 4;
}

template <typename T, int D, int MODE>
static int launch_gather_t(const GatherParams& p, hipStream_t st) {
  const int split = gather_split(p);
  const dim3 grid((unsigned)((p.tiles + 4 / split - 1) / (4 / split))), block(256);
  if (split == 1) hipLaunchKernelGGL((na3d_gather_kernel<T, D, MODE, 1>), grid, block, 0, st, p);
  else if (split == 2) hipLaunchKernelGGL((na3d_gather_kernel<T, D, MODE, 2>), grid, block, 0, st, p);
  else hipLaunchKernelGGL((na3d_gather_kernel<T, D, MODE, 4>), grid, block, 0, st, p);
  return check_launch("na3d_gather_kernel");
}

template <typename T, int MODE>
static int launch_gather_d(const GatherParams& p, hipStream_t st) {
  switch (p.D) {
    case 32: return launch_gather_t<T, 32, MODE>(p, st);
    case 64: return launch_gather_t<T, 64, MODE>(p, st);
    default: return launch_gather_t<T, 128, MODE>(p, st);
  }
}

int launch_gather(const GatherParams& p, int mode, bool is_bf16, hipStream_t st) {
  if (mode == GATHER_FWD) return launch_gather_d<float, GATHER_FWD>(p, st);
  if (mode == GATHER_DQ)
    return is_bf16 ? launch_gather_d<bf16, GATHER_DQ>(p, st) : launch_gather_d<float, GATHER_DQ>(p, st);
  return is_bf16 ? launch_gather_d<bf16, GATHER_DKV>(p, st) : launch_gather_d<float, GATHER_DKV>(p, st);
}

}  // namespace strata
