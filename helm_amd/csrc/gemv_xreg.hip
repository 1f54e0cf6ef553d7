// gemv_xreg.hip — linears of 3 <= M <= 16 tokens with x^T held in registers.
//
// y = fp16(s * (x . q^T) + bias) (int8 weights) or fp16(x . w^T + bias) (fp16
// weights), fp32 accumulation on the matrix cores, with the optional RMSNorm
// prologue, residual add and SwiGLU epilogue of the decode GEMVs.
//
// What bounds it: the weight stream from HBM (M <= 16 products per weight are
// cheap on the matrix cores).  x^T must therefore never cost memory traffic per
// weight tile.  Read from L2 per 16-row tile it moves 2 M bytes of x per 16 bytes
// of weights, and in LDS all of x fits only up to K = 4096 at 16 tokens; here
// every wave keeps the x^T operands of its own k slice in registers for the whole
// launch (80 registers for K = 5120 over eight waves):
//   * one 512-thread workgroup per CU walks 16-row tiles (row tile t, t + grid,
//     ...); its eight waves split K in units of 128 bytes per row;
//   * weights go global -> LDS (16-byte copies, 8 rows x 128 contiguous bytes an
//     instruction) through a private ring of kDepth units per wave, waited for by
//     count: no barrier and no register holds weights in flight, 96 KB per CU;
//   * a unit is read back in the MFMA operand layout (XOR-swizzled chunks, every
//     bank once), int8 turned to fp16 by the exact bias trick;
//   * SwiGLU tiles are eight gate rows and the same eight rows of up, one MFMA tile;
//   * the waves' 16 x 16 partial tiles meet in a double-buffered LDS area, one
//     LDS-only barrier per tile; the waves take turns at the epilogue, so the
//     others' streams never stop.  Scales and biases of the workgroup's rows are
//     staged in LDS at the start: a load in the loop would drain the ring.
// Longer K (int8 only): workgroup b takes k slice b % S of S, fp32 partial sums
// go to the caller's workspace and a second kernel adds them and applies the
// epilogue.
// Measured, weights rotating through HBM: 5120 -> 2 x 17408 with norm and SwiGLU at 12
// tokens 344 -> 36.5 us (4.9 TB/s), 17408 -> 5120 at 8 tokens 32.8 -> 22.9 us, fp16 4096 ->
// 151936 at 4 tokens 221 -> 189 us (6.6 TB/s).  Between two sizes of one shape the rate is 6.9 TB/s;
// 5-9 us of a launch are its start (x from L2: 160 KB per CU at 16 tokens) and end.
#include <algorithm>
#include <type_traits>

#include "helm_common.h"

namespace {

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void_t;

constexpr int kW = 8;                 // waves per workgroup
constexpr int kUnitBytes = 128;       // bytes of one row in a unit
constexpr int kUnitLds = 16 * kUnitBytes;
constexpr int kDepth = 6;             // units of a wave in flight (8 measured equal or 2-3% slower)
constexpr int kPre = 2;               // of these, requested ahead of x (0 equal, 4 or 6 1-4% slower)
constexpr int kMaxTiles = 64;         // row tiles a workgroup may walk (staged scales)

enum { XE_PLAIN = 0, XE_SWIGLU = 1, XE_PART = 2 };

struct XregArgs {
  const uint16_t* x;
  int64_t ldx;
  const uint16_t* norm_w;
  float eps;
  const uint8_t* w;
  const uint8_t* w2;        // SwiGLU: up weights (w holds gate)
  uint32_t ldw;             // bytes
  const uint16_t* scale;
  const uint16_t* scale2;
  const uint16_t* bias;
  const uint16_t* residual;
  uint16_t* y;
  int64_t ldy;
  float* part;              // XE_PART: [S][M][np] partial sums
  int np;
  int M, N, K;
  int S;                    // k slices (1 unless XE_PART)
};

// Waits until at most n of this wave's vector memory operations are outstanding.
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
  asm volatile("" ::: "memory");
}

// One wave's 1 KiB global -> LDS copy: lane l moves 16 bytes from base + off to
// LDS byte lds + 16 l.  Inline assembly so that the compiler does not count it:
// it would wait for every copy in flight before each LDS read.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"   // m0 is named as clobbered on purpose
__device__ __forceinline__ void copy_to_lds(const uint8_t* base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt"
               :
               : "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(off), "s"(base)
               : "memory", "m0");
}
#pragma clang diagnostic pop

// UW: units per wave of one k slice.  EPI: XE_*.
template <bool I8, int UW, bool NORM, int EPI>
__global__ __launch_bounds__(kW * 64) void xreg_gemv_kernel(XregArgs a) {
  constexpr bool SWI = EPI == XE_SWIGLU;
  constexpr int TR = SWI ? 8 : 16;                 // output rows of a tile
  constexpr int kUnitK = I8 ? 128 : 64;            // k of one unit
  constexpr int XV = I8 ? 4 : 2;                   // 8-half x operands per unit
  constexpr bool kScaled = I8 && EPI != XE_PART;
  __shared__ __attribute__((aligned(1024))) uint8_t s_w[kW][kDepth * kUnitLds];
  __shared__ __attribute__((aligned(16))) f4_t s_c[2][kW][64];
  __shared__ float s_ss[NORM ? kW : 1][16];
  __shared__ float s_scale[kScaled ? kMaxTiles * 16 : 1];
  __shared__ float s_bias[EPI == XE_PLAIN ? kMaxTiles * 16 : 1];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int col = lane & 15;       // weight row of a tile (A operand) / token (B operand)
  const int grp = lane >> 4;       // k group of the operands
  const int M = a.M, N = a.N, K = a.K;

  // this workgroup's k slice and row tiles, this wave's units [u0, u1) of the slice
  const int sl = EPI == XE_PART ? (int)blockIdx.x % a.S : 0;
  const int tb = EPI == XE_PART ? (int)blockIdx.x / a.S : (int)blockIdx.x;
  const int nb = EPI == XE_PART ? (int)gridDim.x / a.S : (int)gridDim.x;
  const int tiles = (N + TR - 1) / TR;
  const int T = tb < tiles ? (tiles - 1 - tb) / nb + 1 : 0;
  const int units = (K + kUnitK - 1) / kUnitK;
  const int sa = sl * units / a.S, sn = (sl + 1) * units / a.S - sa;
  const int u0 = sa + wave * sn / kW, u1 = sa + (wave + 1) * sn / kW;   // at most UW of them

  // Copy j of a unit: rows 8 j + lane / 8; LDS chunk lane % 8 of the row holds
  // logical chunk (lane % 8) ^ swz(row), so that the 16 rows one operand read
  // touches lie in different banks.  Chunks past K re-read the row's last one
  // (their x operands are zero), rows past N the last row (not stored).
  const int lrow = lane >> 3;
  const uint32_t kbytes = (uint32_t)K * (I8 ? 1u : 2u);
  uint32_t coff[2];     // byte of this lane's chunk in the wave's first unit
#pragma unroll
  for (int j = 0; j < 2; ++j)
    coff[j] = (uint32_t)u0 * kUnitBytes + (((lane & 7) ^ (((8 * j + lrow) >> 1) & 7)) << 4);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_void_t*)&s_w[wave][0];
  int s_issue = 0;      // ring slot of the next copy
  auto issue = [&](int t, int u) {      // unit u of tile t
    const int r0 = (tb + t * nb) * TR;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      // SwiGLU tiles: eight gate rows, then the same eight rows of up
      const uint32_t row = (uint32_t)min(r0 + (SWI ? 0 : 8 * j) + lrow, N - 1);
      const uint32_t kb = min(coff[j] + (uint32_t)u * kUnitBytes, kbytes - 16);
      copy_to_lds(SWI && j == 1 ? a.w2 : a.w, row * a.ldw + kb, lds0 + s_issue * kUnitLds + j * 1024);
    }
    s_issue = s_issue + 1 == kDepth ? 0 : s_issue + 1;
  };
  // unit n of the wave's stream; units past the end are not requested
  auto issue_nth = [&](int n) {
    if (n / UW < T) issue(n / UW, n % UW);
  };
#pragma unroll
  for (int n = 0; n < kPre; ++n) issue_nth(n);

  // x^T operands of this wave's units: token col, 8 halves each; zero past M and K
  h8_t xr[UW][XV];
  auto xk = [&](int u, int i) {     // first k of operand i of unit u
    return (u0 + u) * kUnitK + (I8 ? (i >> 1) * 64 + grp * 16 + (i & 1) * 8 : i * 32 + grp * 8);
  };
  const uint16_t* xrow = a.x + (int64_t)min(col, M - 1) * a.ldx;
#pragma unroll
  for (int u = 0; u < UW; ++u)
#pragma unroll
    for (int i = 0; i < XV; ++i) xr[u][i] = *reinterpret_cast<const h8_t*>(xrow + min(xk(u, i), K - 8));
  h8_t nw[NORM ? UW : 1][XV];
  if constexpr (NORM) {
#pragma unroll
    for (int u = 0; u < UW; ++u)
#pragma unroll
      for (int i = 0; i < XV; ++i)
        nw[u][i] = *reinterpret_cast<const h8_t*>(a.norm_w + min(xk(u, i), K - 8));
  }
  // scales and biases of the workgroup's rows, two of each per thread
  constexpr int kStg = kMaxTiles * 16 / (kW * 64);
  float scr[kStg], bir[kStg];
#pragma unroll
  for (int k = 0; k < kStg; ++k) {
    const int i = tid + k * kW * 64;
    const int n = (int)min((int64_t)(tb + (int64_t)(i >> 4) * nb) * TR + (i & (TR - 1)), (int64_t)N - 1);
    scr[k] = kScaled ? h2f((SWI && (i & 8) ? a.scale2 : a.scale)[n]) : 0.f;
    bir[k] = EPI == XE_PLAIN && a.bias ? h2f(a.bias[n]) : 0.f;
  }
  // x has arrived: from here on the ring fills while the prologue computes
#pragma unroll
  for (int u = 0; u < UW; ++u)
#pragma unroll
    for (int i = 0; i < XV; ++i) {
      asm volatile("" : "+v"(xr[u][i]));
      if constexpr (NORM) asm volatile("" : "+v"(nw[u][i]));
    }
#pragma unroll
  for (int k = 0; k < kStg; ++k) {
    if constexpr (kScaled) asm volatile("" : "+v"(scr[k]));
    if constexpr (EPI == XE_PLAIN) asm volatile("" : "+v"(bir[k]));
  }
#pragma unroll
  for (int n = kPre; n < kDepth; ++n) issue_nth(n);
#pragma unroll
  for (int k = 0; k < kStg; ++k) {
    if constexpr (kScaled) s_scale[tid + k * kW * 64] = scr[k];
    if constexpr (EPI == XE_PLAIN) s_bias[tid + k * kW * 64] = bir[k];
  }
#pragma unroll
  for (int u = 0; u < UW; ++u)
#pragma unroll
    for (int i = 0; i < XV; ++i)
      if (col >= M || u0 + u >= u1 || xk(u, i) >= K) xr[u][i] = h8_t{};
  if constexpr (NORM) {
    // xn = fp16(w * fp16(x * rsqrt(mean(x^2) + eps))): a lane's share of its token's
    // squares, the four k groups of the wave, then the eight waves through LDS.
    // Every workgroup normalises all tokens, so the instructions per element
    // count: one mixed fma for a square, one for a product and its rounding, half a
    // packed multiply (fp16 x fp16 rounded once, as the fp32 form rounds).
    float s8[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < UW; ++u)
#pragma unroll
      for (int i = 0; i < XV; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float f = (float)xr[u][i][e];
          s8[e] = __builtin_fmaf(f, f, s8[e]);
        }
    float ss = ((s8[0] + s8[1]) + (s8[2] + s8[3])) + ((s8[4] + s8[5]) + (s8[6] + s8[7]));
    ss += __shfl_xor(ss, 16, 64);
    ss += __shfl_xor(ss, 32, 64);
    if (grp == 0) s_ss[wave][col] = ss;
    lds_barrier();
    float tot = 0.f;
#pragma unroll
    for (int w = 0; w < kW; ++w) tot += s_ss[w][col];
    const float rs = rsqrtf(tot / (float)K + a.eps);
    float nz = -0.f;      // x * rs + -0 = x * rs: the mixed fma rounds to fp16 at once
    asm volatile("" : "+v"(nz));
#pragma unroll
    for (int u = 0; u < UW; ++u)
#pragma unroll
      for (int i = 0; i < XV; ++i) {
        h8_t t;
#pragma unroll
        for (int e = 0; e < 8; ++e) t[e] = (_Float16)__builtin_fmaf((float)xr[u][i][e], rs, nz);
        // k past K or another wave's: stays zero whatever the norm weight holds
        xr[u][i] = (u0 + u >= u1 || xk(u, i) >= K) ? h8_t{} : t * nw[u][i];
      }
  }
  lds_barrier();        // staged scales and biases

  int s_read = 0;
  const uint8_t* ring = &s_w[wave][0];
  const int total = T * UW;
  for (int t = 0; t < T; ++t) {
    f4_t c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < UW; ++u) {
      constexpr int kRest = 2 * (kDepth - 1);
      // unit landed: at most the copies of the kDepth - 1 later units outstanding
      // (the stream's end, where fewer follow, waits for all)
      if (t * UW + u + kDepth <= total) wait_vm<kRest>();
      else wait_vm<0>();
      const uint8_t* p = ring + s_read * kUnitLds + col * kUnitBytes;
      uint4 wv[2];
#pragma unroll
      for (int st = 0; st < 2; ++st)
        wv[st] = *reinterpret_cast<const uint4*>(p + (((st * 4 + grp) ^ ((col >> 1) & 7)) << 4));
      s_read = s_read + 1 == kDepth ? 0 : s_read + 1;
      // the slot is refilled once this wave's reads have returned
      asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(wv[0].x), "+v"(wv[0].y), "+v"(wv[0].z), "+v"(wv[0].w),
                   "+v"(wv[1].x), "+v"(wv[1].y), "+v"(wv[1].z), "+v"(wv[1].w) :: "memory");
      if (t + (u + kDepth) / UW < T) issue(t + (u + kDepth) / UW, (u + kDepth) % UW);
      // fp16 weights may be infinite, and 0 * inf is not 0: a unit that is not this
      // wave's is left out (int8 weights times its zero x operands add 0)
      if (!I8 && u0 + u >= u1) continue;
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        if constexpr (I8) {
          h2_t d[8];
          i8x4_to_h2x2(wv[st].x, d[0], d[1]);
          i8x4_to_h2x2(wv[st].y, d[2], d[3]);
          i8x4_to_h2x2(wv[st].z, d[4], d[5]);
          i8x4_to_h2x2(wv[st].w, d[6], d[7]);
          const h8_t a0 = {d[0][0], d[0][1], d[1][0], d[1][1], d[2][0], d[2][1], d[3][0], d[3][1]};
          const h8_t a1 = {d[4][0], d[4][1], d[5][0], d[5][1], d[6][0], d[6][1], d[7][0], d[7][1]};
          c = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, xr[u][2 * st], c, 0, 0, 0);
          c = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, xr[u][2 * st + 1], c, 0, 0, 0);
        } else {
          c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, wv[st]), xr[u][st], c, 0, 0, 0);
        }
      }
    }
    // c[r] = this wave's share of C[row grp * 4 + r][token col]
    f4_t (*sc)[64] = s_c[t & 1];
    sc[wave][lane] = c;
    lds_barrier();      // buffer t & 1 is written again only after tile t + 1's barrier
    if (wave == (t & (kW - 1))) {
      f4_t v = sc[0][lane], vu = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 1; w < kW; ++w) {
        const f4_t o = sc[w][lane];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] += o[r];
      }
      if constexpr (SWI) {   // up rows sit two lane groups above their gate rows
#pragma unroll
        for (int r = 0; r < 4; ++r) vu[r] = __shfl(v[r], (lane + 32) & 63, 64);
      }
      const int n0 = (tb + t * nb) * TR + grp * 4;
      if (col < M && n0 < N && (!SWI || grp < 2)) {
        if constexpr (EPI == XE_PART) {
          // np is N rounded up to a multiple of 4: whole 16-byte stores
          *reinterpret_cast<f4_t*>(a.part + ((int64_t)sl * M + col) * a.np + n0) = v;
        } else {
          uint16_t* yp = a.y + (int64_t)col * a.ldy + n0;
          uint16_t o[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            if constexpr (EPI == XE_SWIGLU) {
              const float g = h2f(f2h(v[r] * s_scale[t * 16 + grp * 4 + r]));
              const float up = h2f(f2h(vu[r] * s_scale[t * 16 + 8 + grp * 4 + r]));
              o[r] = f2h(h2f(f2h(g / (1.0f + expf(-g)))) * up);
            } else {
              float f = v[r];
              if constexpr (kScaled) f *= s_scale[t * 16 + grp * 4 + r];
              f += s_bias[t * 16 + grp * 4 + r];
              if (a.residual && n0 + r < N) f = h2f(a.residual[(int64_t)col * a.ldy + n0 + r]) + h2f(f2h(f));
              o[r] = f2h(f);
            }
          }
          if (n0 + 4 <= N && (reinterpret_cast<uintptr_t>(yp) & 7u) == 0) {
            *reinterpret_cast<uint2*>(yp) =
                make_uint2((uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16));
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (n0 + r < N) yp[r] = o[r];
          }
        }
      }
    }
  }
}

// Second pass over long K: adds the slices' partial sums of four consecutive
// outputs per thread and applies scale, bias and residual (one rounding to fp16).
__global__ __launch_bounds__(256) void xreg_reduce_kernel(XregArgs a) {
  const int n4 = a.np / 4;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= a.M * n4) return;
  const int m = i / n4;
  const int n0 = (i - m * n4) * 4;
  float v[4] = {0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < a.S; ++s) {
    const float4 p = *reinterpret_cast<const float4*>(a.part + ((int64_t)s * a.M + m) * a.np + n0);
    v[0] += p.x; v[1] += p.y; v[2] += p.z; v[3] += p.w;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = n0 + j;
    if (n >= a.N) break;
    float o = v[j] * h2f(a.scale[n]);
    if (a.bias) o += h2f(a.bias[n]);
    const int64_t yi = (int64_t)m * a.ldy + n;
    if (a.residual) o = h2f(a.residual[yi]) + h2f(f2h(o));
    a.y[yi] = f2h(o);
  }
}

constexpr int kCUs = 256;
constexpr int kMaxUwI8 = 6;     // units per wave: 16 x registers each (int8 weights)
constexpr int kMaxUwF16 = 10;   // 8 each (fp16 weights)

int units_of(int K, bool i8) { return i8 ? (K + 127) / 128 : (K + 63) / 64; }
// units of the busiest wave when `units` are cut into S slices of eight waves
int uw_of(int units, int S) {
  const int sn = (units + S - 1) / S;
  return (sn + kW - 1) / kW;
}

// Ring units the busiest wave walks with S slices: rounds of row tiles x units of a wave.
int64_t walk_of(int N, int units, int S) {
  const int tiles = (N + 15) / 16, nb = std::max(1, kCUs / S);
  return (int64_t)((tiles + nb - 1) / nb) * uw_of(units, S);
}

// k slices for K that one slice does not hold: of the few smallest counts the one
// whose busiest workgroup walks the fewest ring units (rounds of row tiles x units
// per wave, unfilled ones included: they take ring slots too).  More slices than
// that lose although they balance better: 25600 -> 5120 at 4 tokens 29.5 us with
// 5 slices, 33.0 with 8; 17408 -> 5120 22.6 with 3, 24.2 with 4.
int choose_slices(int N, int units) {
  int s0 = 1;
  while (uw_of(units, s0) > kMaxUwI8) ++s0;
  if (s0 == 1) return 1;
  int best = s0;
  for (int s = s0 + 1; s < s0 + 4; ++s)
    if (walk_of(N, units, s) < walk_of(N, units, best)) best = s;
  return best;
}

int grid_blocks(int tiles) {
  return std::max(std::min(tiles, kCUs), (tiles + kMaxTiles - 1) / kMaxTiles);
}

template <bool I8, int UW, bool NORM, int EPI>
void launch_xreg(const XregArgs& a, hipStream_t s) {
  constexpr int tr = EPI == XE_SWIGLU ? 8 : 16;
  const int tiles = (a.N + tr - 1) / tr;
  int blocks;
  if (EPI == XE_PART) {
    const int nb = std::max(std::min(tiles, std::max(1, kCUs / a.S)), 1);
    blocks = nb * a.S;
  } else {
    blocks = grid_blocks(tiles);
  }
  hipLaunchKernelGGL((xreg_gemv_kernel<I8, UW, NORM, EPI>), dim3(blocks), dim3(kW * 64), 0, s, a);
}

template <int UW, int EPI>
void launch_i8_norm(const XregArgs& a, hipStream_t s) {
  if constexpr (EPI != XE_PART) {
    if (a.norm_w) return launch_xreg<true, UW, true, EPI>(a, s);
  }
  launch_xreg<true, UW, false, EPI>(a, s);
}

template <int EPI>
void launch_i8(const XregArgs& a, int uw, hipStream_t s) {
  switch (uw) {
    case 1: return launch_i8_norm<1, EPI>(a, s);
    case 2: return launch_i8_norm<2, EPI>(a, s);
    case 3: return launch_i8_norm<3, EPI>(a, s);
    case 4: return launch_i8_norm<4, EPI>(a, s);
    case 5: return launch_i8_norm<5, EPI>(a, s);
    default: return launch_i8_norm<6, EPI>(a, s);
  }
}

template <int UW>
void launch_f16(const XregArgs& a, hipStream_t s) {
  if (a.norm_w) launch_xreg<false, UW, true, XE_PLAIN>(a, s);
  else launch_xreg<false, UW, false, XE_PLAIN>(a, s);
}

bool common_ok(const void* x, int64_t ldx, const void* norm_w, const void* w, int64_t ldw_bytes,
               int M, int N) {
  if (M < 3 || M > 16 || ldx % 8 != 0 || ldw_bytes % 16 != 0) return false;
  if (!helm::aligned16(x) || !helm::aligned16(w) || (norm_w && !helm::aligned16(norm_w))) return false;
  return (int64_t)N * ldw_bytes < (1ll << 31);     // 32-bit weight offsets
}

}  // namespace

namespace helm {

// Ring units (128 bytes of 16 rows) the busiest wave walks in the int8 form.
int xreg_walk_units(int N, int K) {
  const int units = units_of(K, true);
  return (int)std::min<int64_t>(walk_of(N, units, choose_slices(N, units)), 1 << 30);
}

int64_t xreg_workspace_bytes(int M, int N, int K) {
  if (M < 3 || M > 16 || N < 1 || K < 16 || K % 16 != 0) return 0;
  const int S = choose_slices(N, units_of(K, true));
  return S == 1 ? 0 : (int64_t)S * M * ((N + 3) / 4 * 4) * (int64_t)sizeof(float);
}

bool launch_xreg_int8(const void* x, int64_t ldx, const void* norm_w, float eps, const int8_t* q,
                      int64_t ldq, const void* scale, const void* bias, const void* residual,
                      void* y, int64_t ldy, int M, int N, int K, float* part, int64_t part_bytes,
                      hipStream_t stream) {
  if (!common_ok(x, ldx, norm_w, q, ldq, M, N) || K % 16 != 0) return false;
  const int units = units_of(K, true);
  XregArgs a{};
  a.x = static_cast<const uint16_t*>(x); a.ldx = ldx;
  a.norm_w = static_cast<const uint16_t*>(norm_w); a.eps = eps;
  a.w = reinterpret_cast<const uint8_t*>(q); a.ldw = (uint32_t)ldq;
  a.scale = static_cast<const uint16_t*>(scale); a.bias = static_cast<const uint16_t*>(bias);
  a.residual = static_cast<const uint16_t*>(residual);
  a.y = static_cast<uint16_t*>(y); a.ldy = ldy;
  a.M = M; a.N = N; a.K = K; a.S = 1;
  if (uw_of(units, 1) <= kMaxUwI8) {
    launch_i8<XE_PLAIN>(a, uw_of(units, 1), stream);
    return true;
  }
  if (norm_w || !part || !aligned16(part)) return false;
  a.np = (N + 3) / 4 * 4;
  // the chosen split, or the most slices the workspace holds
  const int64_t fit = part_bytes / ((int64_t)M * a.np * (int64_t)sizeof(float));
  a.S = (int)std::min<int64_t>(choose_slices(N, units), fit);
  if (a.S < 1 || uw_of(units, a.S) > kMaxUwI8) return false;
  a.part = part;
  launch_i8<XE_PART>(a, uw_of(units, a.S), stream);
  hipLaunchKernelGGL(xreg_reduce_kernel, dim3((M * (a.np / 4) + 255) / 256), dim3(256), 0, stream, a);
  return true;
}

bool launch_xreg_swiglu(const void* x, int64_t ldx, const void* norm_w, float eps,
                        const int8_t* q_gate, const void* s_gate, const int8_t* q_up,
                        const void* s_up, int64_t ldq, void* y, int64_t ldy, int M, int N, int K,
                        hipStream_t stream) {
  if (!common_ok(x, ldx, norm_w, q_gate, ldq, M, N) || !aligned16(q_up) || K % 16 != 0) return false;
  const int units = units_of(K, true);
  if (uw_of(units, 1) > kMaxUwI8) return false;
  XregArgs a{};
  a.x = static_cast<const uint16_t*>(x); a.ldx = ldx;
  a.norm_w = static_cast<const uint16_t*>(norm_w); a.eps = eps;
  a.w = reinterpret_cast<const uint8_t*>(q_gate); a.w2 = reinterpret_cast<const uint8_t*>(q_up);
  a.ldw = (uint32_t)ldq;
  a.scale = static_cast<const uint16_t*>(s_gate); a.scale2 = static_cast<const uint16_t*>(s_up);
  a.y = static_cast<uint16_t*>(y); a.ldy = ldy;
  a.M = M; a.N = N; a.K = K; a.S = 1;
  launch_i8<XE_SWIGLU>(a, uw_of(units, 1), stream);
  return true;
}

// Units of 64 k the fp16 form walks at this K: its eight waves walk 2, 4, 8 or 10
// each, whole K or not (the products of units past K are left out, their copies are
// not).  0: beyond its registers.
int xreg_fp16_units(int K) {
  const int uw = uw_of(units_of(K, false), 1);
  return uw > kMaxUwF16 ? 0 : kW * (uw <= 2 ? 2 : uw <= 4 ? 4 : uw <= 8 ? 8 : kMaxUwF16);
}

bool launch_xreg_fp16(const void* x, int64_t ldx, const void* norm_w, float eps, const void* w,
                      int64_t ldw, const void* bias, void* y, int64_t ldy, int M, int N, int K,
                      hipStream_t stream) {
  if (!common_ok(x, ldx, norm_w, w, ldw * 2, M, N) || K % 64 != 0) return false;   // whole units
  const int uw = xreg_fp16_units(K) / kW;
  if (!uw) return false;
  XregArgs a{};
  a.x = static_cast<const uint16_t*>(x); a.ldx = ldx;
  a.norm_w = static_cast<const uint16_t*>(norm_w); a.eps = eps;
  a.w = static_cast<const uint8_t*>(w); a.ldw = (uint32_t)(ldw * 2);
  a.bias = static_cast<const uint16_t*>(bias);
  a.y = static_cast<uint16_t*>(y); a.ldy = ldy;
  a.M = M; a.N = N; a.K = K; a.S = 1;
  if (uw == 2) launch_f16<2>(a, stream);
  else if (uw == 4) launch_f16<4>(a, stream);
  else if (uw == 8) launch_f16<8>(a, stream);
  else launch_f16<10>(a, stream);
  return true;
}

}  // namespace helm
