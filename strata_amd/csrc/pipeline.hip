// Rollout step around the network, for gfx950 (bandwidth-bound gathers).
//
// state_patchify: fp32 state [B, C, Z, Y, X] -> bf16 tokens [B, Tz, Ty, Tx, C*P]
//   (P = pz*py*px), the input normalisation of the pipeline
//   (screamcast/normalization.py:109-123) fused with the patchify of a
//   Conv3d(kernel = stride = patch) patch embedding.
// state_update: bf16 tokens [B, Tz, Ty, Tx, C*P] -> fp32 state [B, C, Z, Y, X],
//   the target denormalisation (normalization.py:102-107) and the mixed
//   state / difference update with the qv floor of MixedPredictionAsymmetric.step
//   (screamcast/model_pipelines.py:631-676).
//
// Both are transposes between the channels-first state and the channels-last
// tokens.  A workgroup takes NX consecutive tokens of one (b, tz, ty) token
// row, i.e. the x range [NX*px*xb, NX*px*(xb + 1)) of the C*pz*py state rows
// under them: state rows are read (or written) as runs of NX*px contiguous
// floats, the NX tokens as one contiguous run of NX*C*P bf16, and LDS holds the
// tokens in their final layout in between.
#include "common.h"

namespace strata {

struct PipeParams {
  const float* state;
  void* tokens;  // bf16, read by state_update
  float* next;
  const float* mean;
  const float* std;
  const int32_t* src;
  const float* clamp;
  int B, C, Cin, Z, Y, X;
  int pz, py, px, Tz, Ty, Tx;
  int order;  // element order within a token (state_update)
  int NX;     // tokens per workgroup
  int nxb;    // workgroups per token row
  int vec;    // token runs move as 4-byte pairs (even C*P, 4-byte aligned tokens)
  int KP;     // wide kernels: LDS elements per token, an odd number of dwords
  int rql;    // wide kernels: log2 of the lanes a state-row run takes (a quad of floats each)
  int pxl;    // wide kernels: log2(px)
  uint32_t mp, my;  // wide kernels: divide by pz * py, by py (fast_div)
};

// n / d for n * d < 2^32 as a multiply-high by fast_magic(d) = ceil(2^32 / d) (0: d is 1).
__device__ __forceinline__ int fast_div(int n, uint32_t magic) { return magic ? (int)__umulhi((uint32_t)n, magic) : n; }
static uint32_t fast_magic(int64_t d) { return d == 1 ? 0u : (uint32_t)((((int64_t)1 << 32) + d - 1) / d); }

constexpr int PIPE_LDS = 48 * 1024;
constexpr int PIPE_THREADS = 256;
constexpr int PIPE_U = 4;  // state-row passes per wave whose loads are in flight together

// Lanes a state-row run of `run` floats takes: run rounded up to a power of two (<= 64).
__device__ __forceinline__ int run_lanes(int run) {
  int l = 1;
  while (l < run) l <<= 1;
  return l;
}

// Element index of (c, dz, dy, dx) within a token.
__device__ __forceinline__ int token_elem(const PipeParams& p, int order, int c, int dz, int dy, int dx) {
  return order == 0 ? ((c * p.pz + dz) * p.py + dy) * p.px + dx : ((dz * p.py + dy) * p.px + dx) * p.C + c;
}

// Copy n bf16 between a token run in global memory and the LDS tile: 16-byte
// pieces when the run is 16-byte aligned and n a multiple of 8, else 4-byte
// pieces when p.vec allows, else single elements.
template <bool TO_LDS>
__device__ __forceinline__ void copy_run(const PipeParams& p, bf16* tile, bf16* g, int n, int tid) {
  if (((uintptr_t)g & 15u) == 0 && (n & 7) == 0) {
    u32x4* t = (u32x4*)tile;
    u32x4* q = (u32x4*)g;
    for (int i = tid; i < n / 8; i += PIPE_THREADS) {
      if (TO_LDS) t[i] = q[i];
      else q[i] = t[i];
    }
  } else if (p.vec) {
    uint32_t* t = (uint32_t*)tile;
    uint32_t* q = (uint32_t*)g;
    for (int i = tid; i < n / 2; i += PIPE_THREADS) {
      if (TO_LDS) t[i] = q[i];
      else q[i] = t[i];
    }
  } else {
    for (int i = tid; i < n; i += PIPE_THREADS) {
      if (TO_LDS) tile[i] = g[i];
      else g[i] = tile[i];
    }
  }
}

__global__ __launch_bounds__(PIPE_THREADS) void state_patchify_kernel(PipeParams p) {
  extern __shared__ __attribute__((aligned(16))) bf16 tile[];  // NX tokens, pipe_lds_bytes(p)
  int w = (int)blockIdx.x;
  const int xb = w % p.nxb;
  w /= p.nxb;
  const int ty = w % p.Ty;
  w /= p.Ty;
  const int tz = w % p.Tz;
  const int b = w / p.Tz;
  const int P = p.pz * p.py * p.px;
  const int K = p.C * P;
  const int tx0 = xb * p.NX;
  const int nt = min(p.NX, p.Tx - tx0);  // tokens of this workgroup
  const int run = nt * p.px;             // floats per state row
  const int rows = p.C * p.pz * p.py;
  const int x0 = tx0 * p.px;
  const int tid = (int)threadIdx.x;

  // state rows (c, dz, dy) -> tile[token][element], normalised, in bf16.  A
  // row's run takes RP lanes (run rounded up to a power of two), so a wave pass
  // covers 64 / RP rows, and a wave issues PIPE_U passes' loads before using them.
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int RP = run_lanes(run), sub = lane / RP, xi = lane - sub * RP;
  const int t = xi / p.px, dx = xi - t * p.px;
  const int step = (PIPE_THREADS / 64) * (64 / RP);  // rows per pass of the workgroup
  for (int r0 = wave * (64 / RP) + sub; r0 < rows + step * (PIPE_U - 1); r0 += step * PIPE_U) {
    float v[PIPE_U];
    int cc[PIPE_U], el[PIPE_U];
#pragma unroll
    for (int u = 0; u < PIPE_U; ++u) {
      const int r = r0 + u * step;
      v[u] = 0.f;
      cc[u] = -1;
      if (r < rows && xi < run) {
        const int dy = r % p.py, dz = (r / p.py) % p.pz, c = r / (p.py * p.pz);
        cc[u] = c;
        el[u] = t * K + token_elem(p, 0, c, dz, dy, dx);
        v[u] = p.state[(((int64_t)b * p.C + c) * p.Z + (tz * p.pz + dz)) * (int64_t)p.Y * p.X +
                       (int64_t)(ty * p.py + dy) * p.X + x0 + xi];
      }
    }
#pragma unroll
    for (int u = 0; u < PIPE_U; ++u) {
      if (cc[u] >= 0) {
        float n = v[u];
        if (p.mean) n = (v[u] - p.mean[cc[u]]) / p.std[cc[u]];
        if (!__builtin_isfinite(v[u])) n = 0.f;
        tile[el[u]] = (bf16)n;
      }
    }
  }
  __syncthreads();
  // tile -> nt contiguous tokens
  bf16* dst = (bf16*)p.tokens + ((((int64_t)b * p.Tz + tz) * p.Ty + ty) * p.Tx + tx0) * K;
  copy_run<false>(p, tile, dst, nt * K, tid);
}

__global__ __launch_bounds__(PIPE_THREADS) void state_update_kernel(PipeParams p) {
#pragma clang fp contract(off)
  extern __shared__ __attribute__((aligned(16))) bf16 tile[];  // NX tokens, pipe_lds_bytes(p)
  int w = (int)blockIdx.x;
  const int xb = w % p.nxb;
  w /= p.nxb;
  const int ty = w % p.Ty;
  w /= p.Ty;
  const int tz = w % p.Tz;
  const int b = w / p.Tz;
  const int P = p.pz * p.py * p.px;
  const int K = p.C * P;
  const int tx0 = xb * p.NX;
  const int nt = min(p.NX, p.Tx - tx0);
  const int run = nt * p.px;
  const int rows = p.C * p.pz * p.py;
  const int x0 = tx0 * p.px;
  const int tid = (int)threadIdx.x;

  // nt contiguous tokens -> tile
  bf16* src = (bf16*)p.tokens + ((((int64_t)b * p.Tz + tz) * p.Ty + ty) * p.Tx + tx0) * K;
  copy_run<true>(p, tile, src, nt * K, tid);
  __syncthreads();
  // tile -> state rows (c, dz, dy), as state_patchify: RP lanes per row, 64 / RP
  // rows per wave pass, PIPE_U passes' state loads issued before any store
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int RP = run_lanes(run), sub = lane / RP, xi = lane - sub * RP;
  const int t = xi / p.px, dx = xi - t * p.px;
  const int step = (PIPE_THREADS / 64) * (64 / RP);
  const int64_t plane = (int64_t)p.Z * p.Y * p.X;
  for (int r0 = wave * (64 / RP) + sub; r0 < rows + step * (PIPE_U - 1); r0 += step * PIPE_U) {
    float prev[PIPE_U];
    int cc[PIPE_U], el[PIPE_U];
    bool add[PIPE_U];
    int64_t sp[PIPE_U];
#pragma unroll
    for (int u = 0; u < PIPE_U; ++u) {
      const int r = r0 + u * step;
      prev[u] = 0.f;
      cc[u] = -1;
      add[u] = false;
      if (r < rows && xi < run) {
        const int dy = r % p.py, dz = (r / p.py) % p.pz, c = r / (p.py * p.pz);
        cc[u] = c;
        el[u] = t * K + token_elem(p, p.order, c, dz, dy, dx);
        sp[u] = (int64_t)(tz * p.pz + dz) * p.Y * p.X + (int64_t)(ty * p.py + dy) * p.X + x0 + xi;
        const int sc = p.src ? p.src[c] : c;  // entries outside [0, Cin) add nothing
        add[u] = sc >= 0 && sc < p.Cin;
        if (add[u]) prev[u] = p.state[((int64_t)b * p.Cin + sc) * plane + sp[u]];
      }
    }
#pragma unroll
    for (int u = 0; u < PIPE_U; ++u) {
      const int c = cc[u];
      if (c >= 0) {
        const float pr = (float)tile[el[u]];
        // denormalise in fp32 (a multiply, then an add, each rounded: the pragma
        // above keeps them from contracting to an fma), round to bf16
        float d = pr;
        if (p.mean) d = pr * p.std[c] + p.mean[c];
        d = (float)(bf16)d;
        if (add[u]) d += prev[u];
        if (p.clamp) {
          const float lo = p.clamp[c];
          if (!__builtin_isnan(lo)) d = d < lo ? lo : d;  // clamp(min=lo): NaN stays NaN
        }
        p.next[((int64_t)b * p.C + c) * plane + sp[u]] = d;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// The same transposes with a quad of state floats per thread (px 1, 2 or 4, X a
// multiple of 4, 16-byte aligned state): what bounds the kernels above is the
// index arithmetic and the normalisation's set-up per element (64-bit addresses,
// divisions by py and pz, two table loads), not memory; a quad shares it, and
// moves as one 16-byte load or store.  The token pitch in LDS is an odd number of
// dwords, so a quad's neighbours along x (other tokens) fall on other banks.
// [6,80,16,64,64], us: patchify of patch 1 91 -> 40, 2 x 2 137 -> 47, the
// 2 x 2 x 2 update 171 -> 89 (a torch copy of the state: 35).
// ---------------------------------------------------------------------------

// Copy nt tokens of K bf16 (row pitch ldg in global memory) to or from the LDS
// tile: 16-byte pieces where `by8` allows, else 4-byte pairs (p.vec), else singles.
template <bool TO_LDS>
__device__ __forceinline__ void copy_tokens(bf16* tile, int KP, bf16* g, int64_t ldg, int K, int nt, bool by8, bool by2,
                                            int tid) {
  if (by8) {
    const int per = K / 8, n = nt * per;
    const uint32_t m = per == 1 ? 0u : 0xffffffffu / (uint32_t)per + 1u;
    for (int i = tid; i < n; i += PIPE_THREADS) {
      const int t = fast_div(i, m), k = i - t * per;
      uint32_t* l = (uint32_t*)(tile + t * KP) + 4 * k;
      u32x4* q = (u32x4*)(g + t * ldg) + k;
      if (TO_LDS) {
        const u32x4 v = *q;
#pragma unroll
        for (int e = 0; e < 4; ++e) l[e] = v[e];
      } else {
        *q = (u32x4){l[0], l[1], l[2], l[3]};
      }
    }
  } else if (by2) {
    const int per = K / 2, n = nt * per;
    for (int i = tid; i < n; i += PIPE_THREADS) {
      const int t = i / per, k = i - t * per;
      uint32_t* l = (uint32_t*)(tile + t * KP) + k;
      uint32_t* q = (uint32_t*)(g + t * ldg) + k;
      if (TO_LDS) *l = *q;
      else *q = *l;
    }
  } else {
    for (int i = tid; i < nt * K; i += PIPE_THREADS) {
      const int t = i / K, k = i - t * K;
      if (TO_LDS) tile[t * KP + k] = g[t * ldg + k];
      else g[t * ldg + k] = tile[t * KP + k];
    }
  }
}

// The input normalisation of one value (RunningNorm2d.forward; non-finite inputs 0).
__device__ __forceinline__ float norm_in(float v, bool on, float m, float sd) {
  const float n = on ? (v - m) / sd : v;
  return __builtin_isfinite(v) ? n : 0.f;
}

__global__ __launch_bounds__(PIPE_THREADS) void state_patchify_wide_kernel(PipeParams p) {
  extern __shared__ __attribute__((aligned(16))) bf16 tile[];
  int w = (int)blockIdx.x;
  const int xb = w % p.nxb;
  w /= p.nxb;
  const int ty = w % p.Ty;
  w /= p.Ty;
  const int tz = w % p.Tz, b = w / p.Tz;
  const int K = p.C * p.pz * p.py * p.px, rows = p.C * p.pz * p.py;
  const int tx0 = xb * p.NX, nt = min(p.NX, p.Tx - tx0), run = nt * p.px;
  const int tid = (int)threadIdx.x, x = 4 * (tid & ((1 << p.rql) - 1)), rr = tid >> p.rql, step = PIPE_THREADS >> p.rql;
  const int t = x >> p.pxl, dx = x & (p.px - 1);
  const int64_t YX = (int64_t)p.Y * p.X, ZYX = YX * p.Z;
  const float* src = p.state + b * p.C * ZYX + (int64_t)tz * p.pz * YX + (int64_t)ty * p.py * p.X + tx0 * p.px + x;
  if (x < run) {
    for (int r0 = rr; r0 < rows; r0 += step * PIPE_U) {
      f32x4 v[PIPE_U];
      float m[PIPE_U], sd[PIPE_U];
#pragma unroll
      for (int u = 0; u < PIPE_U; ++u) {
        const int r = min(r0 + u * step, rows - 1);  // a repeated last row is harmless
        const int c = fast_div(r, p.mp), q = r - c * p.pz * p.py, dz = fast_div(q, p.my), dy = q - dz * p.py;
        v[u] = *(const f32x4*)(src + c * ZYX + dz * YX + (int64_t)dy * p.X);
        m[u] = p.mean ? p.mean[c] : 0.f;
        sd[u] = p.mean ? p.std[c] : 1.f;
      }
#pragma unroll
      for (int u = 0; u < PIPE_U; ++u) {
        const int r = min(r0 + u * step, rows - 1);
        float n[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) n[e] = norm_in(v[u][e], p.mean, m[u], sd[u]);
        bf16* d = tile + t * p.KP + r * p.px + dx;
        if (p.px == 1) {
#pragma unroll
          for (int e = 0; e < 4; ++e) d[e * p.KP] = (bf16)n[e];
        } else {  // two pairs: of two tokens (px 2) or of one (px 4)
          *(uint32_t*)d = pack_bf16x2(n[0], n[1]);
          *(uint32_t*)(d + (p.px == 2 ? p.KP : 2)) = pack_bf16x2(n[2], n[3]);
        }
      }
    }
  }
  __syncthreads();
  bf16* dst = (bf16*)p.tokens + ((((int64_t)b * p.Tz + tz) * p.Ty + ty) * p.Tx + tx0) * K;
  copy_tokens<false>(tile, p.KP, dst, K, K, nt, K % 8 == 0 && ((uintptr_t)dst & 15u) == 0, p.vec, tid);
}

__global__ __launch_bounds__(PIPE_THREADS) void state_update_wide_kernel(PipeParams p) {
#pragma clang fp contract(off)
  extern __shared__ __attribute__((aligned(16))) bf16 tile[];
  int w = (int)blockIdx.x;
  const int xb = w % p.nxb;
  w /= p.nxb;
  const int ty = w % p.Ty;
  w /= p.Ty;
  const int tz = w % p.Tz, b = w / p.Tz;
  const int K = p.C * p.pz * p.py * p.px, rows = p.C * p.pz * p.py;
  const int tx0 = xb * p.NX, nt = min(p.NX, p.Tx - tx0), run = nt * p.px;
  const int tid = (int)threadIdx.x, x = 4 * (tid & ((1 << p.rql) - 1)), rr = tid >> p.rql, step = PIPE_THREADS >> p.rql;
  bf16* tok = (bf16*)p.tokens + ((((int64_t)b * p.Tz + tz) * p.Ty + ty) * p.Tx + tx0) * K;
  copy_tokens<true>(tile, p.KP, tok, K, K, nt, K % 8 == 0 && ((uintptr_t)tok & 15u) == 0, p.vec, tid);
  __syncthreads();
  if (x >= run) return;
  const int64_t YX = (int64_t)p.Y * p.X, ZYX = YX * p.Z;
  const int64_t at = (int64_t)tz * p.pz * YX + (int64_t)ty * p.py * p.X + tx0 * p.px + x;
  int el[4];  // token elements of the quad, less the row's part
#pragma unroll
  for (int e = 0; e < 4; ++e)
    el[e] = ((x + e) >> p.pxl) * p.KP + ((x + e) & (p.px - 1)) * (p.order == 0 ? 1 : p.C);
  for (int r0 = rr; r0 < rows; r0 += step * PIPE_U) {
    f32x4 prev[PIPE_U];
#pragma unroll
    for (int u = 0; u < PIPE_U; ++u) {
      const int r = min(r0 + u * step, rows - 1);
      const int c = fast_div(r, p.mp), q = r - c * p.pz * p.py, dz = fast_div(q, p.my), dy = q - dz * p.py;
      const int sc = p.src ? p.src[c] : c;  // entries outside [0, Cin) add nothing
      prev[u] = (f32x4){0.f, 0.f, 0.f, 0.f};
      if (sc >= 0 && sc < p.Cin)
        prev[u] = *(const f32x4*)(p.state + ((int64_t)b * p.Cin + sc) * ZYX + at + dz * YX + (int64_t)dy * p.X);
    }
#pragma unroll
    for (int u = 0; u < PIPE_U; ++u) {
      const int r = r0 + u * step;
      if (r >= rows) break;
      const int c = fast_div(r, p.mp), q = r - c * p.pz * p.py, dz = fast_div(q, p.my), dy = q - dz * p.py;
      const int sc = p.src ? p.src[c] : c;
      const bool add = sc >= 0 && sc < p.Cin;
      const float m = p.mean ? p.mean[c] : 0.f, sd = p.mean ? p.std[c] : 1.f;
      const float floor = p.clamp ? p.clamp[c] : __builtin_nanf("");
      const bf16* tr = tile + (p.order == 0 ? r * p.px : (dz * p.py + dy) * p.px * p.C + c);
      f32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float d = (float)tr[el[e]];
        if (p.mean) d = d * sd + m;  // a multiply, then an add, each rounded (as state_update_kernel)
        d = (float)(bf16)d;
        if (add) d += prev[u][e];
        if (!__builtin_isnan(floor)) d = d < floor ? floor : d;  // clamp(min=floor): NaN stays NaN
        o[e] = d;
      }
      *(f32x4*)(p.next + ((int64_t)b * p.C + c) * ZYX + at + dz * YX + (int64_t)dy * p.X) = o;
    }
  }
}

// The wide kernels' conditions and geometry (p as pipe_setup left it): state
// rows in quads, as many tokens as 20 KiB of LDS hold (eight workgroups per CU),
// a power of two of them.
static bool pipe_wide(PipeParams& p, const float* a, const float* b) {
  if ((p.px != 1 && p.px != 2 && p.px != 4) || p.X % 4 || ((uintptr_t)a & 15u) || ((uintptr_t)b & 15u)) return false;
  const int64_t K = (int64_t)p.C * p.pz * p.py * p.px, KP = (((K + 1) / 2) | 1) * 2;
  int nx = 64 / p.px;
  while (nx * p.px > 4 && nx * KP * 2 > 20480) nx /= 2;
  if (nx * KP * 2 > 64 * 1024) return false;
  while (nx * p.px > 4 && nx / 2 >= p.Tx) nx /= 2;
  p.pxl = p.px == 1 ? 0 : p.px == 2 ? 1 : 2;
  p.rql = 0;
  while (4 << p.rql < nx * p.px) ++p.rql;
  p.KP = (int)KP;
  p.NX = nx;
  p.nxb = (p.Tx + nx - 1) / nx;
  p.mp = fast_magic((int64_t)p.pz * p.py);
  p.my = fast_magic(p.py);
  return (int64_t)p.C * p.pz * p.py * p.pz * p.py < ((int64_t)1 << 32) &&
         (int64_t)p.B * p.Tz * p.Ty * p.nxb <= 0x7fffffff;
}

// ---------------------------------------------------------------------------
// Dealiased patchify: the low-passes along y and x of dealias_axis_kernel and the
// patchify in one pass, bit for bit as that chain (normalise, filter along y, then
// along x, each sum in tap order, fp32).  A workgroup takes a run of channel
// slices (c, dz), four token rows and up to 128 columns: the rows its taps
// reach are read once, normalised, into LDS; the y sums go to LDS; the x sums go
// as bf16 into the token tile, which leaves like the patchify's.  The chain moved
// the fp32 state five times; this reads it once (the taps' rows overlap in L2).
// Bound by its instructions (VALU 88% busy: the exact division of the normalisation, twice per
// element; the taps through LDS).  [6,80,16,64,64], patch 2 x 2, 5 taps: 367 us in
// three launches -> 113.
// ---------------------------------------------------------------------------
// Per workgroup: four token rows, and channel slices for up to 64 elements of a
// token in 40 KiB of LDS (four workgroups per CU or more).  Two or eight rows and 16 to
// 128 elements measured 109-125 us at the shape above, patch 2 x 2 and 4 x 4.
constexpr int DEALIAS_ROWS = 4, DEALIAS_KC = 64, DEALIAS_LDS = 40 * 1024;

struct DealiasTokens {
  PipeParams p;
  int CB, ncb;      // channel slices per workgroup, such runs
  int NTY, nyb;     // token rows per workgroup, such runs
  int ny, nx;       // taps (1: no filter along the axis)
  int SR, XW;       // LDS rows per slice, floats per LDS row
  uint32_t mXW4, mSR, mRows;  // fast_div by XW / 4, SR, NTY * py
  float fy[16], fx[16];
};

// NT: the taps of both axes at compile time (their reads go out together and the
// filter stays in scalar registers), 0: any counts.
template <int NT>
__global__ __launch_bounds__(PIPE_THREADS) void dealias_patchify_kernel(DealiasTokens d) {
  if constexpr (NT > 0) d.ny = d.nx = NT;
  extern __shared__ __attribute__((aligned(16))) float dl[];
  const PipeParams& p = d.p;
  // one XCD takes neighbours: their tokens share lines, their rows overlap
  int w = xcd_tile_order((int)gridDim.x, (int)__builtin_amdgcn_workgroup_id_x());
  const int cb = w % d.ncb;
  w /= d.ncb;
  const int xb = w % p.nxb;
  w /= p.nxb;
  const int yb = w % d.nyb;
  w /= d.nyb;
  const int tz = w % p.Tz, b = w / p.Tz;
  const int slices = p.C * p.pz, s0 = cb * d.CB, ns = min(d.CB, slices - s0);
  const int ty0 = yb * d.NTY, nty = min(d.NTY, p.Ty - ty0), tx0 = xb * p.NX, nt = min(p.NX, p.Tx - tx0);
  const int rows = d.NTY * p.py, run = nt * p.px, xo = tx0 * p.px;
  const int loy = (d.ny - 1) / 2, lox = (d.nx - 1) / 2;
  // source rows [r0, r0 + nr) and columns [c0, c0 + nc) (c0, nc multiples of 4)
  auto clampi = [](int v, int hi) { return min(max(v, 0), hi); };
  const int r0 = d.ny == 1 ? ty0 * p.py : clampi(p.py * ty0 - loy, p.Y - p.py);
  const int r1 = d.ny == 1 ? (ty0 + nty) * p.py
                           : clampi(p.py * (ty0 + nty - 1) - loy + d.ny - 1, p.Y - p.py) + p.py;
  const int c0 = (d.nx == 1 ? xo : clampi(xo - lox, p.X - p.px)) & ~3;
  const int c1 = d.nx == 1 ? xo + run : clampi(xo + run - p.px - lox + d.nx - 1, p.X - p.px) + p.px;
  const int nr = r1 - r0, nq = (c1 - c0 + 3) / 4, XQ = d.XW / 4;
  float* A = dl;                              // [CB][SR][XW] normalised state
  float* G = A + d.CB * d.SR * d.XW;          // [CB][rows][XW] filtered along y
  bf16* tile = (bf16*)(G + d.CB * rows * d.XW);
  const int tid = (int)threadIdx.x;
  const int64_t YX = (int64_t)p.Y * p.X, ZYX = YX * p.Z;

  for (int i0 = tid; i0 < ns * d.SR * XQ; i0 += PIPE_THREADS * PIPE_U) {
    f32x4 v[PIPE_U];
    int at[PIPE_U], cc[PIPE_U];
#pragma unroll
    for (int k = 0; k < PIPE_U; ++k) {
      const int i = i0 + k * PIPE_THREADS, row = fast_div(i, d.mXW4), q = i - row * XQ, s = fast_div(row, d.mSR),
                r = row - s * d.SR;
      at[k] = -1;
      if (s >= ns || q >= nq || r >= nr) continue;
      const int dz = s0 + s - fast_div(s0 + s, p.mp) * p.pz;
      cc[k] = fast_div(s0 + s, p.mp);
      at[k] = row * d.XW + 4 * q;
      v[k] = *(const f32x4*)(p.state + ((int64_t)b * p.C + cc[k]) * ZYX + (int64_t)(tz * p.pz + dz) * YX +
                             (int64_t)(r0 + r) * p.X + c0 + 4 * q);
    }
#pragma unroll
    for (int k = 0; k < PIPE_U; ++k) {
      if (at[k] < 0) continue;
      const float m = p.mean ? p.mean[cc[k]] : 0.f, sd = p.mean ? p.std[cc[k]] : 1.f;
      f32x4 n;
#pragma unroll
      for (int e = 0; e < 4; ++e) n[e] = norm_in(v[k][e], p.mean, m, sd);
      *(f32x4*)(A + at[k]) = n;
    }
  }
  __syncthreads();
  for (int i = tid; i < ns * rows * XQ; i += PIPE_THREADS) {
    const int row = fast_div(i, d.mXW4), q = i - row * XQ, s = fast_div(row, d.mRows), yo = row - s * rows;
    const int j = ty0 + fast_div(yo, p.my), u = yo - (j - ty0) * p.py;
    if (q >= nq || j >= ty0 + nty) continue;
    const float* a = A + s * d.SR * d.XW + 4 * q;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (d.ny == 1) {
      acc = *(const f32x4*)(a + yo * d.XW);
    } else {
#pragma unroll
      for (int t = 0; t < (NT ? NT : d.ny); ++t) {
        const f32x4 v = *(const f32x4*)(a + (clampi(p.py * j - loy + t, p.Y - p.py) + u - r0) * d.XW);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = fmaf(d.fy[t], v[e], acc[e]);
      }
      if (d.nx > 1) {  // the x pass takes non-finite values as 0
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = __builtin_isfinite(acc[e]) ? acc[e] : 0.f;
      }
    }
    *(f32x4*)(G + row * d.XW + 4 * q) = acc;
  }
  __syncthreads();
  const int RQ = 1 << p.rql;
  for (int i = tid; i < ns * rows * RQ; i += PIPE_THREADS) {
    const int row = i >> p.rql, x = 4 * (i & (RQ - 1)), s = fast_div(row, d.mRows), yo = row - s * rows;
    const int jr = fast_div(yo, p.my), u = yo - jr * p.py;
    if (x >= run || jr >= nty) continue;
    const float* g = G + row * d.XW - c0;  // indexed by the state's column
    float o[4];
    if (d.nx == 1) {
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = g[xo + x + e];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = 0.f;
      // Column i reads clamp(px (i / px) - lox + t) + i % px: i - lox + t where no
      // tap is clamped, so a quad slides one window; else each column its own.
      const int xa = xo + x, ja = xa & ~(p.px - 1), jb = (xa + 3) & ~(p.px - 1);
      if (ja - lox >= 0 && jb - lox + d.nx - 1 <= p.X - p.px) {
        float w0 = g[xa - lox], w1 = g[xa - lox + 1], w2 = g[xa - lox + 2];
#pragma unroll
        for (int t = 0; t < (NT ? NT : d.nx); ++t) {
          const float w3 = g[xa - lox + t + 3];
          o[0] = fmaf(d.fx[t], w0, o[0]);
          o[1] = fmaf(d.fx[t], w1, o[1]);
          o[2] = fmaf(d.fx[t], w2, o[2]);
          o[3] = fmaf(d.fx[t], w3, o[3]);
          w0 = w1;
          w1 = w2;
          w2 = w3;
        }
      } else {
#pragma unroll
        for (int t = 0; t < (NT ? NT : d.nx); ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int ia = xa + e, jx = ia & ~(p.px - 1);
            o[e] = fmaf(d.fx[t], g[clampi(jx - lox + t, p.X - p.px) + ia - jx], o[e]);
          }
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t = (x + e) >> p.pxl, dx = (x + e) & (p.px - 1);
      const float v = __builtin_isfinite(o[e]) ? o[e] : 0.f;
      tile[(jr * p.NX + t) * p.KP + (s * p.py + u) * p.px + dx] = (bf16)v;
    }
  }
  __syncthreads();
  const int K = slices * p.py * p.px, Kc = ns * p.py * p.px, k0 = s0 * p.py * p.px;
  for (int j = 0; j < nty; ++j) {
    bf16* dst = (bf16*)p.tokens + ((((int64_t)b * p.Tz + tz) * p.Ty + ty0 + j) * p.Tx + tx0) * K + k0;
    copy_tokens<false>(tile + j * p.NX * p.KP, p.KP, dst, K, Kc, nt,
                       K % 8 == 0 && Kc % 8 == 0 && ((uintptr_t)dst & 15u) == 0, p.vec && Kc % 2 == 0 && k0 % 2 == 0, tid);
  }
}

// LDS of one workgroup: NX tokens of C*P bf16, rounded up to 16 bytes (sized
// to the need so that small tokens leave room for many workgroups per CU).
static size_t pipe_lds_bytes(const PipeParams& p) {
  return ((size_t)p.NX * p.C * p.pz * p.py * p.px * 2 + 15) / 16 * 16;
}

// Shared validation and launch geometry.  Returns OK and fills p, or an error.
static int pipe_setup(PipeParams& p, const char* name, int B, int C, const int32_t* grid, const int32_t* patch) {
  const std::string n(name);
  if (B < 0 || C <= 0) return fail(STRATA_HIP_EINVAL, n + ": bad batch/channels");
  static const char* axis = "zyx";
  for (int a = 0; a < 3; ++a) {
    if (grid[a] <= 0 || patch[a] <= 0)
      return fail(STRATA_HIP_EINVAL, n + ": grid and patch sizes must be positive on axis " + axis[a]);
    if (grid[a] % patch[a] != 0)
      return fail(STRATA_HIP_EINVAL, n + ": grid not a multiple of the patch on axis " + axis[a]);
  }
  p.B = B;
  p.C = C;
  p.Z = grid[0];
  p.Y = grid[1];
  p.X = grid[2];
  p.pz = patch[0];
  p.py = patch[1];
  p.px = patch[2];
  p.Tz = p.Z / p.pz;
  p.Ty = p.Y / p.py;
  p.Tx = p.X / p.px;
  const int64_t K = (int64_t)C * p.pz * p.py * p.px;
  if (K * 2 > PIPE_LDS)
    return fail(STRATA_HIP_EUNSUPPORTED, n + ": a token of C*pz*py*px elements must fit 48 KiB of bf16");
  if (p.px > 64) return fail(STRATA_HIP_EUNSUPPORTED, n + ": patch width above 64");
  // up to 64 state floats per row run (a lane each), as many tokens as LDS holds
  int NX = (int)(PIPE_LDS / (K * 2));
  const int nx_run = 64 / p.px > 1 ? 64 / p.px : 1;
  NX = NX < nx_run ? NX : nx_run;
  // at most 16 KiB when that still leaves 16 tokens: more workgroups per CU
  if (NX > 16 && (int64_t)NX * K * 2 > 16384) NX = (int)(16384 / (K * 2)) > 16 ? (int)(16384 / (K * 2)) : 16;
  NX = NX < p.Tx ? NX : p.Tx;
  p.NX = NX;
  p.nxb = (p.Tx + NX - 1) / NX;
  const int64_t blocks = (int64_t)B * p.Tz * p.Ty * p.nxb;
  if (blocks > 0x7fffffff || (int64_t)B * C * p.Z * p.Y * p.X > ((int64_t)1 << 40))
    return fail(STRATA_HIP_EUNSUPPORTED, n + ": problem too large for one launch");
  return STRATA_HIP_OK;
}

// One axis pass of the dealiasing low-pass (see strata_hip_dealias_axis).  The
// tensor is viewed as [outer, S, inner] around the filtered axis.  A wave owns
// DEALIAS_LPW lines and its lanes step through the lines' contiguous floats, so
// every index below the lane level is wave-uniform (scalar registers, no
// per-thread division), and the lines' loads of one tap are issued together:
//   x axis (inner = 1): a line is one row of S floats; output i of the row
//     reads its taps along the row;
//   y, z axes: a line is (o, i), the `inner` floats of output row i; its taps
//     are the rows clamp(P*(i/P) - lo + t, 0, S - P) + i%P of the same o.
struct DealiasParams {
  const float* src;
  float* dst;
  const float* mean;
  const float* std;
  int64_t lines;  // x: outer rows; y, z: outer * S
  int64_t inner;  // stride of the axis in floats
  int64_t cdiv;   // lines (x) or outer index (y, z) per channel step: c = (. / cdiv) % C
  int C, S, P, lo, taps;
  float f[16];
};

constexpr int DEALIAS_LPW = 8;  // lines per wave, their loads of one tap issued together

template <bool XAXIS>
__global__ __launch_bounds__(256) void dealias_axis_kernel(DealiasParams p) {
  constexpr int R = DEALIAS_LPW;
  const int64_t line0 = ((int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * R;
  const int lane = threadIdx.x & 63;
  if (line0 >= p.lines) return;  // uniform per wave
  const float* src[R];
  float* dst[R];
  float m[R], sd[R];
  int j0[R], u[R];
  bool live[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t line = line0 + r < p.lines ? line0 + r : p.lines - 1;  // a repeated last line is harmless
    live[r] = line0 + r < p.lines;
    int64_t o = line;  // x: the row; y, z: the outer index
    int irow = 0;      // y, z: the output row
    if constexpr (!XAXIS) {
      o = line / p.S;
      irow = (int)(line - o * p.S);
    }
    m[r] = 0.f;
    sd[r] = 1.f;
    if (p.mean) {
      const int c = (int)((o / p.cdiv) % p.C);
      m[r] = p.mean[c];
      sd[r] = p.std[c];
    }
    if constexpr (XAXIS) {
      src[r] = p.src + line * p.S;
      dst[r] = p.dst + line * p.S;
    } else {
      j0[r] = p.P * (irow / p.P) - p.lo;
      u[r] = irow % p.P;
      src[r] = p.src + o * p.S * p.inner;
      dst[r] = p.dst + line * p.inner;
    }
  }
  const int64_t n = XAXIS ? p.S : p.inner;
  for (int64_t k = lane; k < n; k += 64) {
    int xj0 = 0, xu = 0;
    if constexpr (XAXIS) {
      xj0 = p.P * ((int)k / p.P) - p.lo;
      xu = (int)k % p.P;
    }
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.f;
    for (int t = 0; t < p.taps; ++t) {
      float v[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if constexpr (XAXIS)
          v[r] = src[r][min(max(xj0 + t, 0), p.S - p.P) + xu];
        else
          v[r] = src[r][(int64_t)(min(max(j0[r] + t, 0), p.S - p.P) + u[r]) * p.inner + k];
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        float nv = v[r];
        if (p.mean) nv = (v[r] - m[r]) / sd[r];
        if (!__builtin_isfinite(v[r])) nv = 0.f;
        acc[r] = fmaf(p.f[t], nv, acc[r]);
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (live[r]) dst[r][k] = acc[r];
  }
}

}  // namespace strata

using namespace strata;

extern "C" int strata_hip_dealias_axis(const strata_hip_dealias_axis_args* a, void* stream) {
  if (!a) return fail(STRATA_HIP_EINVAL, "dealias_axis: null args");
  if (!a->src || !a->dst) return fail(STRATA_HIP_EINVAL, "dealias_axis: null tensor pointer");
  if ((a->mean == nullptr) != (a->std == nullptr))
    return fail(STRATA_HIP_EINVAL, "dealias_axis: mean and std must both be given or both be NULL");
  if (a->batch < 0 || a->channels <= 0) return fail(STRATA_HIP_EINVAL, "dealias_axis: bad batch/channels");
  if (a->grid[0] <= 0 || a->grid[1] <= 0 || a->grid[2] <= 0) return fail(STRATA_HIP_EINVAL, "dealias_axis: bad grid");
  if (a->axis < 0 || a->axis > 2) return fail(STRATA_HIP_EINVAL, "dealias_axis: axis must be 0, 1 or 2");
  const int S = a->grid[a->axis];
  if (a->patch <= 0 || S % a->patch != 0)
    return fail(STRATA_HIP_EINVAL, "dealias_axis: patch must be positive and divide the grid on the axis");
  if (a->taps < 1 || a->taps > 16) return fail(STRATA_HIP_EINVAL, "dealias_axis: taps must be in 1..16");
  if (a->src == a->dst) return fail(STRATA_HIP_EINVAL, "dealias_axis: src and dst must not alias");
  DealiasParams p = {};
  p.src = a->src;
  p.dst = a->dst;
  p.mean = a->mean;
  p.std = a->std;
  p.C = a->channels;
  p.S = S;
  p.P = a->patch;
  p.taps = a->taps;
  p.lo = (a->taps - 1) / 2;
  for (int t = 0; t < a->taps; ++t) p.f[t] = a->filter[t];
  const int64_t Z = a->grid[0], Y = a->grid[1], X = a->grid[2];
  const int64_t total = (int64_t)a->batch * a->channels * Z * Y * X;
  if (total == 0) return STRATA_HIP_OK;
  if (total > ((int64_t)1 << 40)) return fail(STRATA_HIP_EUNSUPPORTED, "dealias_axis: problem too large");
  // [outer, S, inner] around the axis; cdiv: outer indices (y, z) or rows (x) per channel
  p.inner = a->axis == 2 ? 1 : (a->axis == 1 ? X : Y * X);
  const int64_t outer = total / (S * p.inner);
  p.lines = a->axis == 2 ? outer : outer * S;
  p.cdiv = a->axis == 0 ? 1 : (a->axis == 1 ? Z : Z * Y);
  const int64_t blocks = (p.lines + 4 * DEALIAS_LPW - 1) / (4 * DEALIAS_LPW);
  if (blocks > 0x7fffffff) return fail(STRATA_HIP_EUNSUPPORTED, "dealias_axis: problem too large for one launch");
  if (a->axis == 2)
    hipLaunchKernelGGL(dealias_axis_kernel<true>, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, p);
  else
    hipLaunchKernelGGL(dealias_axis_kernel<false>, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, p);
  return check_launch("dealias_axis_kernel");
}

extern "C" int strata_hip_state_patchify(const strata_hip_state_patchify_args* a, void* stream) {
  if (!a) return fail(STRATA_HIP_EINVAL, "state_patchify: null args");
  PipeParams p = {};
  const int rc = pipe_setup(p, "state_patchify", a->batch, a->channels, a->grid, a->patch);
  if (rc != STRATA_HIP_OK) return rc;
  if (!a->state || !a->tokens) return fail(STRATA_HIP_EINVAL, "state_patchify: null tensor pointer");
  if ((a->mean == nullptr) != (a->std == nullptr))
    return fail(STRATA_HIP_EINVAL, "state_patchify: mean and std must both be given or both be NULL");
  p.state = a->state;
  p.tokens = a->tokens;
  p.mean = a->mean;
  p.std = a->std;
  p.vec = (p.C * p.pz * p.py * p.px) % 2 == 0 && ((uintptr_t)a->tokens & 3u) == 0;
  const bool wide = pipe_wide(p, a->state, a->state);
  const int64_t blocks = (int64_t)p.B * p.Tz * p.Ty * p.nxb;
  if (blocks == 0) return STRATA_HIP_OK;
  if (wide) {
    hipLaunchKernelGGL(state_patchify_wide_kernel, dim3((unsigned)blocks), dim3(PIPE_THREADS),
                       (size_t)p.NX * p.KP * 2, (hipStream_t)stream, p);
    return check_launch("state_patchify_wide_kernel");
  }
  hipLaunchKernelGGL(state_patchify_kernel, dim3((unsigned)blocks), dim3(PIPE_THREADS), pipe_lds_bytes(p),
                     (hipStream_t)stream, p);
  return check_launch("state_patchify_kernel");
}

extern "C" int strata_hip_state_update(const strata_hip_state_update_args* a, void* stream) {
  if (!a) return fail(STRATA_HIP_EINVAL, "state_update: null args");
  PipeParams p = {};
  const int rc = pipe_setup(p, "state_update", a->batch, a->channels, a->grid, a->patch);
  if (rc != STRATA_HIP_OK) return rc;
  if (!a->pred || !a->next) return fail(STRATA_HIP_EINVAL, "state_update: null tensor pointer");
  if (a->order != 0 && a->order != 1) return fail(STRATA_HIP_EINVAL, "state_update: order must be 0 or 1");
  if ((a->mean == nullptr) != (a->std == nullptr))
    return fail(STRATA_HIP_EINVAL, "state_update: mean and std must both be given or both be NULL");
  // Without a channel map every channel is a difference of the same state channel.
  if (!a->src_channel && a->state_channels < a->channels)
    return fail(STRATA_HIP_EINVAL, "state_update: state has fewer channels than the prediction");
  if (a->state_channels < 0 || (a->state_channels > 0) != (a->state != nullptr))
    return fail(STRATA_HIP_EINVAL, "state_update: state and state_channels must both be given or both be empty");
  p.tokens = const_cast<void*>(a->pred);
  p.state = a->state;
  p.next = a->next;
  p.mean = a->mean;
  p.std = a->std;
  p.src = a->src_channel;
  p.clamp = a->clamp_min;
  p.Cin = a->state_channels;
  p.order = a->order;
  p.vec = (p.C * p.pz * p.py * p.px) % 2 == 0 && ((uintptr_t)a->pred & 3u) == 0;
  const bool wide = pipe_wide(p, a->state, a->next);
  const int64_t blocks = (int64_t)p.B * p.Tz * p.Ty * p.nxb;
  if (blocks == 0) return STRATA_HIP_OK;
  if (wide) {
    hipLaunchKernelGGL(state_update_wide_kernel, dim3((unsigned)blocks), dim3(PIPE_THREADS), (size_t)p.NX * p.KP * 2,
                       (hipStream_t)stream, p);
    return check_launch("state_update_wide_kernel");
  }
  hipLaunchKernelGGL(state_update_kernel, dim3((unsigned)blocks), dim3(PIPE_THREADS), pipe_lds_bytes(p),
                     (hipStream_t)stream, p);
  return check_launch("state_update_kernel");
}

extern "C" int strata_hip_dealias_patchify(const strata_hip_state_patchify_args* a, const float* taps_y, int32_t ny,
                                           const float* taps_x, int32_t nx, void* stream) {
  if (!a) return fail(STRATA_HIP_EINVAL, "dealias_patchify: null args");
  if (ny < 1 || ny > 16 || nx < 1 || nx > 16) return fail(STRATA_HIP_EINVAL, "dealias_patchify: taps must be in 1..16");
  if ((ny > 1 && !taps_y) || (nx > 1 && !taps_x)) return fail(STRATA_HIP_EINVAL, "dealias_patchify: null taps");
  DealiasTokens d = {};
  PipeParams& p = d.p;
  const int rc = pipe_setup(p, "dealias_patchify", a->batch, a->channels, a->grid, a->patch);
  if (rc != STRATA_HIP_OK) return rc;
  if (!a->state || !a->tokens) return fail(STRATA_HIP_EINVAL, "dealias_patchify: null tensor pointer");
  if ((a->mean == nullptr) != (a->std == nullptr))
    return fail(STRATA_HIP_EINVAL, "dealias_patchify: mean and std must both be given or both be NULL");
  if ((p.px != 1 && p.px != 2 && p.px != 4) || p.X % 4 || ((uintptr_t)a->state & 15u))
    return fail(STRATA_HIP_EUNSUPPORTED,
                "dealias_patchify: patch widths 1, 2 and 4, an x extent that is a multiple of 4 and a 16-byte aligned "
                "state (else strata_hip_dealias_axis per axis and strata_hip_state_patchify)");
  // No filter: the chain is the patchify alone, whose kernel has no LDS passes over the state
  // and keeps what the normalisation overflows (the filters take it as 0).
  if (ny == 1 && nx == 1) return strata_hip_state_patchify(a, stream);
  p.state = a->state;
  p.tokens = a->tokens;
  p.mean = a->mean;
  p.std = a->std;
  d.ny = ny;
  d.nx = nx;
  for (int t = 0; t < ny; ++t) d.fy[t] = ny > 1 ? taps_y[t] : 1.f;
  for (int t = 0; t < nx; ++t) d.fx[t] = nx > 1 ? taps_x[t] : 1.f;
  // up to 128 columns, in equal runs of whole quads and tokens
  const int unit = 4 > p.px ? 4 : p.px, nch = (p.X + 127) / 128;
  const int runx = ((p.X + nch - 1) / nch + unit - 1) / unit * unit;
  p.NX = runx / p.px;
  p.nxb = (p.Tx + p.NX - 1) / p.NX;
  p.pxl = p.px == 1 ? 0 : p.px == 2 ? 1 : 2;
  while (4 << p.rql < runx) ++p.rql;
  d.NTY = DEALIAS_ROWS;
  if (d.NTY > p.Ty) d.NTY = p.Ty;
  d.nyb = (p.Ty + d.NTY - 1) / d.NTY;
  d.CB = 1;
  while (d.CB * p.py * p.px < DEALIAS_KC) d.CB *= 2;
  const int slices = p.C * p.pz, rows = d.NTY * p.py;
  d.SR = rows + (ny > 1 ? ny - 1 : 0);
  const int wide = runx + (nx > 1 ? nx - 1 : 0) + 6;  // the aligned start and end
  d.XW = (wide < p.X + 3 ? wide : p.X + 3) / 4 * 4;
  auto lds = [&]() {
    p.KP = ((d.CB * p.py * p.px + 1) / 2 | 1) * 2;
    return (size_t)d.CB * (d.SR + rows) * d.XW * 4 + (size_t)d.NTY * p.NX * p.KP * 2;
  };
  while (d.CB > 1 && (lds() > DEALIAS_LDS || d.CB / 2 >= slices)) d.CB /= 2;
  if (lds() > 64 * 1024) return fail(STRATA_HIP_EUNSUPPORTED, "dealias_patchify: patch or filter too large");
  d.ncb = (slices + d.CB - 1) / d.CB;
  d.mXW4 = fast_magic(d.XW / 4);
  d.mSR = fast_magic(d.SR);
  d.mRows = fast_magic(rows);
  p.mp = fast_magic(p.pz);
  p.my = fast_magic(p.py);
  p.vec = (slices * p.py * p.px) % 2 == 0 && ((uintptr_t)a->tokens & 3u) == 0;
  const int64_t blocks = (int64_t)p.B * p.Tz * d.nyb * p.nxb * d.ncb;
  if (blocks == 0) return STRATA_HIP_OK;
  if (blocks > 0x7fffffff) return fail(STRATA_HIP_EUNSUPPORTED, "dealias_patchify: problem too large for one launch");
  const dim3 grid((unsigned)blocks), block(PIPE_THREADS);
  hipStream_t st = (hipStream_t)stream;
  switch (ny == nx ? ny : 0) {
    case 2: hipLaunchKernelGGL(dealias_patchify_kernel<2>, grid, block, lds(), st, d); break;
    case 3: hipLaunchKernelGGL(dealias_patchify_kernel<3>, grid, block, lds(), st, d); break;
    case 4: hipLaunchKernelGGL(dealias_patchify_kernel<4>, grid, block, lds(), st, d); break;
    case 5: hipLaunchKernelGGL(dealias_patchify_kernel<5>, grid, block, lds(), st, d); break;
    default: hipLaunchKernelGGL(dealias_patchify_kernel<0>, grid, block, lds(), st, d); break;
  }
  return check_launch("dealias_patchify_kernel");
}
