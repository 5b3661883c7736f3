// Weight gradient of the GEMM backward for gfx950:  dW[n, k] = sum_m g[m, n] x[m, k]
//
// g [M, N] is the output gradient and x [M, K] the input, both rows contiguous, so
// the contraction runs down the rows of both: neither MFMA operand is contiguous
// along it.  A stage of 64 rows of a 256-column panel of each streams into LDS as
// it lies (buffer_load ... lds, 512 bytes per row) and the fragments are read
// transposed (ds_read_b64_tr_b16: 4 rows of one column per lane).  With x as the
// MFMA's A operand a lane of v_mfma_f32_16x16x32_bf16 owns four consecutive k of
// one n, a 16-byte store.
//
// dW has few 256 x 256 tiles (36 for 3072 x 768) and a long contraction, so the rows
// are split over enough workgroups to fill the chip (one per CU), each writes an
// fp32 partial and a second launch adds the partials in split order: the order of
// every addition is fixed by the shape, the result repeats bit for bit.
//
// With a bias gradient (the column sums of g) each of a row range's workgroups along
// k sums its share of the stages, 4 more MFMAs beside 32 there (a ones operand
// against the g fragments it holds anyway); the partials, [splits * kt, N] fp32, are
// added in the second launch: at [65536, 3072] 11 us more here in the place of a 39 us
// pass over g of its own.
//
// Bound by the copies and LDS reads beside the MFMAs, as the forward's 256 x 256
// kernel (same tile, ring and burst split): at [65536, 3072] x [65536, 768] the matrix
// cores are busy 52% of the time, the LDS reads 38%, waves wait 33%.  Against the library's product, us:
// [65536, N] x [65536, K] of N x K = 3072 x 768 433 -> 292, 2304 x 768 526 -> 233,
// 768 x 768 272 -> 89; M = 131072, 4096 x 1024 1236 -> 869 (1265 TFLOP/s); at M =
// 1000 both are launch-bound.
#include "common.h"

namespace strata {

struct WgradParams {
  const bf16* g;
  const bf16* x;
  float* part;  // [splits, N, K] fp32, or null: one split, straight to out
  float* bpart; // [splits * kt, N] fp32 column sums of g, or null
  bf16* out;    // [N, K]
  int64_t M, N, K, ldg, ldx;
  int nt, kt;   // 256-wide tiles along N and K
  int splits, rows;  // row ranges, rows per range (a multiple of 64)
};

constexpr int WG_BK = 64;                    // rows per stage
constexpr int WG_HALF = WG_BK * 512;         // bytes of one panel's stage
constexpr int WG_STAGE = 2 * WG_HALF;

template <bool BIAS>
__global__ __launch_bounds__(512, 1) void weight_grad_kernel(WgradParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int NW = 8, LPW = WG_HALF / 1024 / NW;  // 1-KiB copies per wave, panel and stage
  __shared__ __attribute__((aligned(1024))) char lds[2 * WG_STAGE];
  const int tid = (int)__builtin_amdgcn_workitem_id_x();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, n16 = lane & 15, g4 = lane >> 4;
  const int wk = wave >> 2, wn = wave & 3;  // wave tile: 128 k x 64 n
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;

  // The tiles of one row range on one XCD: they read the same rows of g and x.
  int w = xcd_tile_order((int)gridDim.x, (int)__builtin_amdgcn_workgroup_id_x());
  const int tk = w % p.kt;
  w /= p.kt;
  const int tn = w % p.nt, sp = w / p.nt;
  const int64_t k0 = (int64_t)tk * 256, n0 = (int64_t)tn * 256;
  const int64_t m0 = (int64_t)sp * p.rows;
  const int rows = (int)min((int64_t)p.rows, p.M - m0);
  const int nk = (rows + WG_BK - 1) / WG_BK;

  // Copy j of a panel's stage fills rows 2c, 2c + 1 (c = j * NW + wave), 32 lanes of 16
  // bytes each; the chunk a lane fetches is swizzled by the row (two chunks at a time,
  // so that the transposed reads of 16 rows x 16 columns are free of bank conflicts).
  // Columns past the matrix read as zero.
  uint32_t vx[LPW], vg[LPW];
#pragma unroll
  for (int j = 0; j < LPW; ++j) {
    const int row = 2 * (j * NW + wave) + (lane >> 5), c = (lane & 31) ^ ((row & 7) << 1);
    vx[j] = k0 + 8 * c < p.K ? (uint32_t)(row * p.ldx * 2 + c * 16) : OOB;
    vg[j] = n0 + 8 * c < p.N ? (uint32_t)(row * p.ldg * 2 + c * 16) : OOB;
  }
  const char* xb = (const char*)(p.x + m0 * p.ldx + k0);
  const char* gb = (const char*)(p.g + m0 * p.ldg + n0);
  auto issue = [&](int kt, int slot, bool is_g) {
    const int left = rows - kt * WG_BK;  // rows of the stage that exist
    const u32x4 r = make_rsrc(is_g ? gb + (int64_t)kt * WG_BK * p.ldg * 2 : xb + (int64_t)kt * WG_BK * p.ldx * 2, OOB);
    const uint32_t dst = lds_base + slot * WG_STAGE + (is_g ? WG_HALF : 0) + wave * 1024;
#pragma unroll
    for (int j = 0; j < LPW; ++j) {
      uint32_t vo = is_g ? vg[j] : vx[j];
      if (left < WG_BK && 2 * (j * NW + wave) + (lane >> 5) >= left) vo = OOB;
      dma_row16(r, dst + j * NW * 1024, vo);
    }
  };

  // Transposed fragment reads: lane (n16, g4) addresses row 4 g4 + (n16 >> 2), columns
  // 4 (n16 & 3) of a 16-column block, and receives rows 4 g4 .. + 3 of column n16.
  const int tr = 4 * g4 + (n16 >> 2);
  auto frag_off = [&](int col) {  // byte offset of a 16-column block, rows 0 .. 15 (row & 7 repeats every 8)
    const int c = col / 8 + ((n16 & 3) >> 1);
    return (uint32_t)(tr * 512 + ((c ^ ((tr & 7) << 1)) << 4) + 8 * (n16 & 1));
  };
  uint32_t ao[8], bo[4];
#pragma unroll
  for (int i = 0; i < 8; ++i) ao[i] = frag_off(128 * wk + 16 * i);
#pragma unroll
  for (int j = 0; j < 4; ++j) bo[j] = WG_HALF + frag_off(64 * wn + 16 * j);
  auto frag = [&](const char* st, uint32_t off, int kk) {
    const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_PTR(bf16x4, st + off + kk * 32 * 512));
    const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_PTR(bf16x4, st + off + kk * 32 * 512 + 16 * 512));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };

  f32x4 acc[8][4];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  f32x4 bacc[BIAS ? 4 : 1];
  bf16x8 ones;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = (bf16)1.f;
#pragma unroll
  for (int j = 0; j < (BIAS ? 4 : 1); ++j) bacc[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  int btick = tk;  // stages until this workgroup's next turn at the column sums
  issue(0, 0, false);
  issue(0, 0, true);
  for (int kt = 0; kt < nk; ++kt) {
    const bool mine = BIAS && btick == 0 && wk == 0;  // uniform
    if (BIAS) btick = btick == 0 ? p.kt - 1 : btick - 1;
    wait_vmcnt(0);
    lds_barrier();  // the stage has landed for every wave; the other slot is free
    const int wr = (kt + 1) & 1;
    if (kt + 1 < nk) issue(kt + 1, wr, false);
    const char* st = lds + (kt & 1) * WG_STAGE;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      bf16x8 a[8], b[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = frag(st, bo[j], kk);
#pragma unroll
      for (int i = 0; i < 8; ++i) a[i] = frag(st, ao[i], kk);
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
      if constexpr (BIAS) {
        if (mine) {
#pragma unroll
          for (int j = 0; j < 4; ++j) bacc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, b[j], bacc[j], 0, 0, 0);
        }
      }
      if (kk == 0 && kt + 1 < nk) {
        __builtin_amdgcn_sched_barrier(0);
        issue(kt + 1, wr, true);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (!BIAS) __builtin_amdgcn_iglp_opt(1);
  }

  if constexpr (BIAS) {
    if (wk == 0 && g4 == 0) {  // every row of the ones product holds the sums
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int64_t n = n0 + 64 * wn + 16 * j + n16;
        if (n < p.N) p.bpart[((int64_t)sp * p.kt + tk) * p.N + n] = bacc[j][0];
      }
    }
  }
  // Block (i, j): k = 128 wk + 16 i + 4 g4 + r, n = 64 wn + 16 j + n16.  N and K are
  // multiples of 8: a quad lies inside the matrix or outside it.
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int64_t n = n0 + 64 * wn + 16 * j + n16;
    if (n >= p.N) continue;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int64_t k = k0 + 128 * wk + 16 * i + 4 * g4;
      if (k >= p.K) continue;
      if (p.part) {
        *(f32x4*)(p.part + ((int64_t)sp * p.N + n) * p.K + k) = acc[i][j];
      } else {
        *(u32x2*)(p.out + n * p.K + k) =
            (u32x2){pack_bf16x2(acc[i][j][0], acc[i][j][1]), pack_bf16x2(acc[i][j][2], acc[i][j][3])};
      }
    }
  }
#endif
}

// out = the sum of the partials in split order, eight elements per thread; the last
// blocks the bias gradient's, 16 columns each, 16 threads a column: each adds every
// 16th partial in order, then the 16 sums in order.
__global__ __launch_bounds__(256) void weight_grad_finish_kernel(const float* __restrict__ part, bf16* __restrict__ out,
                                                                 int64_t n, int splits, int blocks,
                                                                 const float* __restrict__ bpart,
                                                                 bf16* __restrict__ bout, int64_t N, int bsplits) {
  if ((int)blockIdx.x >= blocks) {
    __shared__ float red[16][16];
    const int c = threadIdx.x & 15, r = threadIdx.x >> 4;
    const int64_t col = ((int64_t)blockIdx.x - blocks) * 16 + c;
    float s = 0.f;
    if (col < N)
      for (int k = r; k < bsplits; k += 16) s += bpart[(int64_t)k * N + col];
    red[r][c] = s;
    __syncthreads();
    if (r == 0 && col < N) {
      for (int k = 1; k < 16; ++k) s += red[k][c];
      bout[col] = (bf16)s;
    }
    return;
  }
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
  if (i >= n) return;
  f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
  const float* q = part + i;
#pragma unroll 4
  for (int s = 0; s < splits; ++s, q += n) {
    a += *(const f32x4*)q;
    b += *(const f32x4*)(q + 4);
  }
  *(u32x4*)(out + i) = (u32x4){pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3]), pack_bf16x2(b[0], b[1]),
                               pack_bf16x2(b[2], b[3])};
}

// Splits of the rows: one workgroup per CU (the ring admits one), at least four
// stages each.  256, not the device's own count: the order of the sums is the
// shape's alone.  From 129 tiles on one split leaves CUs idle (144 of 256 at
// 6144 x 1536) and more take more rounds and 190 MB of partials; the caller keeps
// such shapes on torch's product where that is faster (ops._weight_grad_pays).
static int wgrad_splits(int64_t m, int64_t n, int64_t k) {
  const int64_t tiles = ((n + 255) / 256) * ((k + 255) / 256), stages = (m + WG_BK - 1) / WG_BK;
  int64_t s = tiles >= 256 ? 1 : 256 / tiles;
  const int64_t most = stages / 4 < 1 ? 1 : stages / 4;
  return (int)(s < most ? s : most);
}

// fp32 elements of the bias partials, a multiple of 4 (the weight partials follow).
static int64_t wgrad_bias_floats(int64_t n, int64_t k, int64_t splits) {
  return (splits * ((k + 255) / 256) * n + 3) / 4 * 4;
}

}  // namespace strata

extern "C" int64_t strata_hip_weight_grad_workspace(int64_t m, int64_t n, int64_t k, int32_t bias) {
  if (m <= 0 || n <= 0 || k <= 0) return 0;
  const int64_t s = strata::wgrad_splits(m, n, k);
  return (s > 1 ? s * n * k : 0) + (bias ? strata::wgrad_bias_floats(n, k, s) : 0);
}

extern "C" int strata_hip_weight_grad(const strata_hip_weight_grad_args* a, void* stream) {
  using namespace strata;
  if (!a) return fail(STRATA_HIP_EINVAL, "weight_grad: null args");
  if (a->m <= 0 || a->n < 0 || a->k < 0) return fail(STRATA_HIP_EINVAL, "weight_grad: bad m/n/k");
  if (a->n > 0 && a->k == 0 && a->bias_out)
    return fail(STRATA_HIP_EINVAL, "weight_grad: no columns of x (the column sums alone: strata_hip_bias_grad)");
  if (a->n == 0 || a->k == 0) return STRATA_HIP_OK;
  if (!a->g || !a->x || !a->out) return fail(STRATA_HIP_EINVAL, "weight_grad: null pointer");
  if (a->n % 8 || a->k % 8 || a->ldg % 8 || a->ldx % 8 || a->ldg < a->n || a->ldx < a->k)
    return fail(STRATA_HIP_EINVAL, "weight_grad: n, k and the row strides must be multiples of 8, rows not overlapping");
  if (((uintptr_t)a->g & 15) || ((uintptr_t)a->x & 15) || ((uintptr_t)a->out & 15) || ((uintptr_t)a->workspace & 15))
    return fail(STRATA_HIP_EINVAL, "weight_grad: g, x, out and workspace must be 16-byte aligned");
  if (64 * a->ldg * 2 + 4096 >= (int64_t)OOB || 64 * a->ldx * 2 + 4096 >= (int64_t)OOB)
    return fail(STRATA_HIP_EUNSUPPORTED, "weight_grad: row strides too long");
  WgradParams p = {};
  p.g = (const bf16*)a->g;
  p.x = (const bf16*)a->x;
  p.out = (bf16*)a->out;
  p.M = a->m;
  p.N = a->n;
  p.K = a->k;
  p.ldg = a->ldg;
  p.ldx = a->ldx;
  p.nt = (int)((a->n + 255) / 256);
  p.kt = (int)((a->k + 255) / 256);
  const int want = wgrad_splits(a->m, a->n, a->k);
  const int64_t stages = (a->m + WG_BK - 1) / WG_BK, per = (stages + want - 1) / want;
  if (per * WG_BK > 0x7fffffff || (int64_t)p.nt * p.kt * want > 0x7fffffff || a->n * a->k / 2048 > 0x7ffffff0)
    return fail(STRATA_HIP_EUNSUPPORTED, "weight_grad: problem too large for one launch");
  p.rows = (int)(per * WG_BK);
  p.splits = (int)((stages + per - 1) / per);  // ranges that hold rows
  const bool bias = a->bias_out != nullptr;
  if (want > 1 || bias) {
    if (!a->workspace) return fail(STRATA_HIP_EINVAL, "weight_grad: null workspace");
    if (bias) p.bpart = a->workspace;
    if (want > 1) p.part = a->workspace + (bias ? wgrad_bias_floats(a->n, a->k, want) : 0);
  }
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)(p.nt * p.kt * p.splits));
  if (bias) hipLaunchKernelGGL(weight_grad_kernel<true>, grid, dim3(512), 0, st, p);
  else hipLaunchKernelGGL(weight_grad_kernel<false>, grid, dim3(512), 0, st, p);
  const int64_t n = a->n * a->k;
  const int blocks = p.part ? (int)((n / 8 + 255) / 256) : 0, bblocks = bias ? (int)((a->n + 15) / 16) : 0;
  if (blocks + bblocks)
    hipLaunchKernelGGL(weight_grad_finish_kernel, dim3((unsigned)(blocks + bblocks)), dim3(256), 0, st, p.part, p.out, n,
                       p.splits, blocks, p.bpart, (bf16*)a->bias_out, a->n, p.splits * p.kt);
  return check_launch("weight_grad kernels");
}
