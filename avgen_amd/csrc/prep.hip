// Operand preparation for the attention kernels: padded copies of the
// sequence tensors and the padded key bias.
//
// The attention kernels stream sequence tiles through LDS with direct
// global->LDS loads.  Two kinds of copy of a (B, H, L, D) strided tensor are
// made here, once per call, each padded with zeros to Lp = L rounded up to a
// whole 64-row tile (transpose_padded_len), so that every tile load is a
// full, branch-free load with loop-invariant per-lane offsets and padded
// positions hold finite values:
//   rows: xr[((b*H + h)*Lp + i)*D + d] = x[b, h, i, d]      (row-major)
//   cols: xt[((b*H + h)*D + d)*Lp + i] = x[b, h, i, d]      (head_dim-major)
// The head_dim-major copy serves the products that contract over the
// sequence (O += P V, dV += P^T dO, dK += dS^T Q, dQ += dS K): their MFMA
// operand then has its k index along a contiguous row and is one 16-byte LDS
// read, instead of transpose reads, which run at a fraction of the rate on
// gfx950.  Each copy is HBM-bound: one read of x, one write per copy.
#include "avattn_device.h"
#include "avattn_kernels.h"

namespace avattn {

// One 64-row tile of x (256 threads): rows s0 .. s0 + 63 of one (b, h) slice
// whose row 0 is at `src`, rotated first when the slice's tables are given
// (the copies then hold the rotated rows src/avgen/models/rope.py:332-338
// produces), to `xr` (row-major, D apart) and / or `xt` (head_dim-major, Lp
// apart; both already at the tile).  Returns the thread's share of the
// largest squared row norm (NORM) and of "every value is finite" (FINITE).
struct TileScan {
  float nmax;
  bool finite;
};
template <int D, bool NORM>
__device__ __forceinline__ TileScan copy_tile(const bf16* __restrict__ src, int64_t sl, int s0, int L, int Lp,
                                              bf16* __restrict__ xr, bf16* __restrict__ xt,
                                              const float* __restrict__ ct, const float* __restrict__ st,
                                              bool check_finite, bf16* tile) {
  constexpr int S = 64;       // sequence rows per tile
  constexpr int CPR = D / 8;  // 16-byte chunks per row
  constexpr int LD = D + 2;   // LDS row pitch in bf16 (odd word count: column reads spread over banks)
  const int tid = threadIdx.x;
  TileScan r{0.f, true};
  // Load 64 rows (zeros past L) as 16-byte chunks; write the row-major copy
  // and scatter into the pitched tile for the head_dim-major one.
#pragma unroll
  for (int i = 0; i < S * CPR / 256; ++i) {
    const int c = tid + i * 256;
    const int row = c / CPR, ch = c % CPR;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (s0 + row < L) {
      v = *reinterpret_cast<const u32x4*>(src + (int64_t)(s0 + row) * sl + ch * 8);
      if (ct) {
        // Channels 8*ch .. +7 are pairs 4*ch .. +3 of row s0 + row.
        const int64_t t = (int64_t)(s0 + row) * (D / 2) + 4 * ch;
        v = rotate8(v, *reinterpret_cast<const f32x4*>(ct + t), *reinterpret_cast<const f32x4*>(st + t), false);
      }
    }
    if (check_finite) {
#pragma unroll
      for (int w = 0; w < 4; ++w)
        r.finite = r.finite && (v[w] & 0x7f80u) != 0x7f80u && (v[w] & 0x7f800000u) != 0x7f800000u;
    }
    if (xr) *reinterpret_cast<u32x4*>(xr + row * D + ch * 8) = v;
    if (xt) {
      uint32_t* dst = reinterpret_cast<uint32_t*>(tile + row * LD + ch * 8);
#pragma unroll
      for (int w = 0; w < 4; ++w) dst[w] = v[w];
    }
    if constexpr (NORM) {
      // A row's CPR chunks sit in CPR consecutive lanes: sum their squares.
      float n = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) n = fmaf(bf16_lo(v[w]), bf16_lo(v[w]), fmaf(bf16_hi(v[w]), bf16_hi(v[w]), n));
#pragma unroll
      for (int off = 1; off < CPR; off <<= 1) n += __shfl_xor(n, off);
      r.nmax = fmaxf(r.nmax, n);
    }
  }
  if (xt) {
    __syncthreads();
    // Each thread writes 16-byte chunks of head_dim-major rows: 8 consecutive
    // sequence positions of one channel.
#pragma unroll
    for (int i = 0; i < D * (S / 8) / 256; ++i) {
      const int c = tid + i * 256;
      const int d = c / (S / 8), j = c % (S / 8);
      u32x4 v;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const uint16_t lo = __builtin_bit_cast(uint16_t, tile[(8 * j + 2 * w) * LD + d]);
        const uint16_t hi = __builtin_bit_cast(uint16_t, tile[(8 * j + 2 * w + 1) * LD + d]);
        v[w] = (uint32_t)lo | ((uint32_t)hi << 16);
      }
      *reinterpret_cast<u32x4*>(xt + (int64_t)d * Lp + 8 * j) = v;
    }
  }
  return r;
}

// Whether every value of a 64-row tile is finite (this thread's share).
template <int D>
__device__ __forceinline__ bool tile_finite(const bf16* __restrict__ src, int64_t sl, int s0, int L) {
  constexpr int CPR = D / 8;
  bool ok = true;
#pragma unroll
  for (int i = 0; i < 64 * CPR / 256; ++i) {
    const int c = threadIdx.x + i * 256;
    const int row = s0 + c / CPR;
    if (row < L) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(src + (int64_t)row * sl + (c % CPR) * 8);
#pragma unroll
      for (int w = 0; w < 4; ++w) ok = ok && (v[w] & 0x7f80u) != 0x7f80u && (v[w] & 0x7f800000u) != 0x7f800000u;
    }
  }
  return ok;
}

// The 64 lanes of a wave as the keys j0 .. j0 + 63 of batch b: which are
// attended (j < Lk and the mask, if any, is nonzero).
__device__ __forceinline__ uint64_t attended_keys(const uint8_t* mask, int64_t msb, int b, int j0, int Lk) {
  const int j = j0 + (threadIdx.x & 63);
  return __builtin_amdgcn_ballot_w64(j < Lk && (mask == nullptr || mask[b * msb + j] != 0));
}

// Key bias and flags of one 64-key tile (threads 0..63): kbias[b*Lkp + j] = 0
// if key j is attended, else -inf; kfull[b*(Lkp/32) + t] = 1 if all 32 keys
// of tile t are attended.
__device__ __forceinline__ void write_key_bias(uint64_t att, int b, int j0, int Lkp, float* __restrict__ kbias,
                                               int* __restrict__ kfull) {
  const int lane = threadIdx.x;
  if (lane >= 64) return;
  kbias[(int64_t)b * Lkp + j0 + lane] = (att >> lane) & 1 ? 0.f : kNegInf;
  if (lane < 2) kfull[(int64_t)b * (Lkp / 32) + j0 / 32 + lane] = (uint32_t)(att >> (32 * lane)) == 0xffffffffu;
}

// Forward preparation, one launch (separate ones cost 4-8 us each at short
// sequences: K, V and key-bias launches 39 us of a 338 us call at
// (2,20,3600,128)).  Workgroups [0, nk): K row copy of one 64-key tile of one
// (b, kv head) with the tile's largest squared row norm in kmax2 (none with
// fp8, whose K copy is launch_quantize_rows); then the V^T copy of one tile
// each, those of kv head 0 also writing the tile's key bias and flags.  A
// tile without an attended key whose k and v are finite is marked in the sign
// bit of its kmax2 (the norm itself is >= 0): it contributes exactly nothing
// and the forward may leave it out.  Leaving such tiles out at both ends here
// and in the backward took 75,600 queries x 512 text keys (one sample of 388
// keys, one of none, 40 heads, D 128, fwd+bwd) from 7.35 to 5.59 ms.
template <int D>
__global__ __launch_bounds__(256) void prep_fwd_kernel(FwdArgs a, int nk) {
  __shared__ bf16 tile[64 * (D + 2)];
  __shared__ float wmax[4];
  __shared__ int wfin[4];
  const int nt = a.Lkp / 64;
  const bool is_k = (int)blockIdx.x < nk;
  const int u = is_k ? blockIdx.x : blockIdx.x - nk;
  const int t = u % nt, bh = u / nt;
  const int b = bh / a.Hkv, h = bh % a.Hkv;
  const int s0 = 64 * t;
  if (is_k) {
    const bool unattended = a.mask != nullptr && attended_keys(a.mask, a.msb, b, s0, a.Lk) == 0;
    const float* ct = a.cos_k ? a.cos_k + b * a.rksb : nullptr;
    const float* st = a.cos_k ? a.sin_k + b * a.rksb : nullptr;
    TileScan r = copy_tile<D, true>(a.k + b * a.ksb + h * a.ksh, a.ksl, s0, a.Lk, a.Lkp,
                                    a.kr + ((int64_t)bh * a.Lkp + s0) * D, nullptr, ct, st, unattended, tile);
    if (unattended) r.finite = r.finite && tile_finite<D>(a.v + b * a.vsb + h * a.vsh, a.vsl, s0, a.Lk);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) r.nmax = fmaxf(r.nmax, __shfl_xor(r.nmax, off));
    const int fin = __all(r.finite);
    if ((threadIdx.x & 63) == 0) {
      wmax[threadIdx.x >> 6] = r.nmax;
      wfin[threadIdx.x >> 6] = fin;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      const bool skip = unattended && wfin[0] && wfin[1] && wfin[2] && wfin[3];
      a.kmax2[(int64_t)bh * nt + t] = __float_as_uint(fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]))) |
                                      (skip ? kTileSkip : 0u);
    }
  } else {
    if (h == 0) write_key_bias(attended_keys(a.mask, a.msb, b, s0, a.Lk), b, s0, a.Lkp, a.kbias, a.kfull);
    copy_tile<D, false>(a.v + b * a.vsb + h * a.vsh, a.vsl, s0, a.Lk, a.Lkp, nullptr,
                        a.vt + (int64_t)bh * D * a.Lkp + s0, nullptr, nullptr, false, tile);
  }
}

// Backward preparation, one launch.  Workgroups in order: one 64-key tile of
// one (b, kv head) each (K^T copy, and without staged dS the K and V row
// copies; those of kv head 0 write the tile's key bias and flags; with a mask
// and staged dS, kskip says whether no key of the tile is attended while its
// k is finite, see key_hull_kernel); then, unless the query side is reused,
// one 64-row tile of one (b, query head) each for the q and dO copies the
// dK/dV kernel needs, and the row statistics: lse2 = lse * log2(e) (+inf for
// -inf and padded rows, whose P is then exactly 0) and ndelta =
// -rowsum(dout * out), kStatRows rows per TPR threads.  Under a mask a row with lse
// -inf attends nothing: its dout and out are not read.
// (One row each, its (b, h, row) by 64-bit divisions, took 485 us for 2 x 40 x
// 75,600 rows of which half are read, against 423.)
constexpr int kStatRows = 4;
template <int D>
__global__ __launch_bounds__(256) void prep_bwd_kernel(BwdArgs a, int nk, int nq, int nd) {
  __shared__ bf16 tile[64 * (D + 2)];
  int u = blockIdx.x;
  if (u < nk) {
    const int nt = a.Lkp / 64;
    const int t = u % nt, bh = u / nt;
    const int b = bh / a.Hkv, h = bh % a.Hkv;
    const int s0 = 64 * t;
    const uint64_t att = attended_keys(a.mask, a.msb, b, s0, a.Lk);
    if (h == 0) write_key_bias(att, b, s0, a.Lkp, a.kbias, a.kfull);
    const float* ct = a.cos_k ? a.cos_k + b * a.rksb : nullptr;
    const float* st = a.cos_k ? a.sin_k + b * a.rksb : nullptr;
    const bool rows = a.ds == nullptr;
    const int64_t row0 = ((int64_t)bh * a.Lkp + s0) * D;
    const bool scan = a.kskip != nullptr && att == 0;
    const TileScan r = copy_tile<D, false>(a.k + b * a.ksb + h * a.ksh, a.ksl, s0, a.Lk, a.Lkp,
                                           rows ? a.kr + row0 : nullptr, a.kt + (int64_t)bh * D * a.Lkp + s0, ct, st,
                                           scan, tile);
    if (rows)
      copy_tile<D, false>(a.v + b * a.vsb + h * a.vsh, a.vsl, s0, a.Lk, a.Lkp, a.vr + row0, nullptr, nullptr,
                          nullptr, false, tile);
    if (a.kskip != nullptr) {
      const int skip = __syncthreads_and(scan && r.finite);
      if (threadIdx.x == 0) a.kskip[(int64_t)bh * nt + t] = skip;
    } else if (a.khull != nullptr && t == 0 && threadIdx.x == 0) {
      a.khull[2 * bh] = 0;
      a.khull[2 * bh + 1] = nt;
    }
    return;
  }
  u -= nk;
  if (u < nq + nd) {
    const bool is_q = u < nq;
    if (!is_q) u -= nq;
    const int nt = a.Lqp / 64;
    const int t = u % nt, bh = u / nt;
    const int b = bh / a.Hq, h = bh % a.Hq;
    const int64_t row0 = ((int64_t)bh * a.Lqp + 64 * t) * D;
    if (is_q)
      copy_tile<D, false>(a.q + b * a.qsb + h * a.qsh, a.qsl, 64 * t, a.Lq, a.Lqp, a.qr + row0, nullptr,
                          a.cos_q ? a.cos_q + b * a.rqsb : nullptr, a.cos_q ? a.sin_q + b * a.rqsb : nullptr, false,
                          tile);
    else
      copy_tile<D, false>(a.dout + b * a.dosb + h * a.dosh, a.dosl, 64 * t, a.Lq, a.Lqp, a.dor + row0, nullptr,
                          nullptr, nullptr, false, tile);
    return;
  }
  u -= nq + nd;
  constexpr int TPR = D / 8;  // threads per row
  constexpr int RPB = 256 / TPR;
  const int nb = (a.Lqp + kStatRows * RPB - 1) / (kStatRows * RPB);
  const int bh = u / nb, i0 = u % nb * (kStatRows * RPB) + threadIdx.x / TPR;
  const int h = bh % a.Hq, b = bh / a.Hq;
  const int c = threadIdx.x % TPR;
  const bf16* dp = a.dout + b * a.dosb + h * a.dosh + 8 * c;
  const bf16* op = a.out + b * a.osb + h * a.osh + 8 * c;
  float l[kStatRows];
  u32x4 x[kStatRows], y[kStatRows];
#pragma unroll
  for (int r = 0; r < kStatRows; ++r) {
    const int i = i0 + r * RPB;
    l[r] = i < a.Lq ? a.lse[(int64_t)bh * a.Lq + i] : kNegInf;
    x[r] = y[r] = u32x4{0u, 0u, 0u, 0u};
    if (i < a.Lq && (a.mask == nullptr || l[r] != kNegInf)) {
      x[r] = *reinterpret_cast<const u32x4*>(dp + (int64_t)i * a.dosl);
      y[r] = *reinterpret_cast<const u32x4*>(op + (int64_t)i * a.osl);
    }
  }
#pragma unroll
  for (int r = 0; r < kStatRows; ++r) {
    float acc = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      acc = fmaf(__uint_as_float(x[r][w] << 16), __uint_as_float(y[r][w] << 16), acc);
      acc = fmaf(__uint_as_float(x[r][w] & 0xffff0000u), __uint_as_float(y[r][w] & 0xffff0000u), acc);
    }
#pragma unroll
    for (int off = TPR / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, TPR);
    const int i = i0 + r * RPB;
    if (i < a.Lqp && c == 0) {
      a.ndelta[(int64_t)bh * a.Lqp + i] = -acc;
      a.lse2[(int64_t)bh * a.Lqp + i] = (l[r] == kNegInf) ? kPosInf : l[r] * kLog2e;
    }
  }
}

// Per (b, kv head), the range [khull[2 p], khull[2 p + 1]) of 64-key tiles
// outside which every tile is marked in kskip (empty when all are).  One wave
// per pair.
__global__ __launch_bounds__(64) void key_hull_kernel(const int* __restrict__ kskip, int nt, int* __restrict__ khull) {
  int lo = nt, hi = 0;
  for (int t = threadIdx.x; t < nt; t += 64) {
    if (kskip[(int64_t)blockIdx.x * nt + t] == 0) {
      lo = min(lo, t);
      hi = max(hi, t + 1);
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    lo = min(lo, __shfl_xor(lo, off));
    hi = max(hi, __shfl_xor(hi, off));
  }
  if (threadIdx.x == 0) {
    khull[2 * blockIdx.x] = lo < hi ? lo : 0;
    khull[2 * blockIdx.x + 1] = hi;
  }
}

hipError_t launch_prep_fwd(const FwdArgs& a, int head_dim, hipStream_t stream) {
  const int64_t tiles = (int64_t)a.B * a.Hkv * (a.Lkp / 64);
  if (2 * tiles > 2147483647) return hipErrorInvalidValue;
  const int nk = a.k8 ? 0 : (int)tiles;
  const dim3 grid((unsigned)(nk + tiles));
  LaunchTimer timer(kKidTranspose, stream);
  if (head_dim == 128)
    hipLaunchKernelGGL(prep_fwd_kernel<128>, grid, dim3(256), 0, stream, a, nk);
  else
    hipLaunchKernelGGL(prep_fwd_kernel<64>, grid, dim3(256), 0, stream, a, nk);
  return hipGetLastError();
}

hipError_t launch_prep_bwd(const BwdArgs& a, int head_dim, hipStream_t stream) {
  const int64_t nk = (int64_t)a.B * a.Hkv * (a.Lkp / 64);
  const int64_t qtiles = (int64_t)a.B * a.Hq * (a.Lqp / 64);
  // Kept from an earlier call (reuse_q): the statistics and a rotated q copy.
  // Copies that rows that overlap need are made again: that call may have read
  // the same values in place, from rows that do not.
  const int64_t nq = a.qt == a.qr && !(a.reuse_q && a.cos_q) ? qtiles : 0, nd = a.dt == a.dor ? qtiles : 0;
  const int rpb = 256 / (head_dim / 8) * kStatRows;
  const int64_t ns = a.reuse_q ? 0 : (int64_t)a.B * a.Hq * ((a.Lqp + rpb - 1) / rpb);
  if (nk + nq + nd + ns > 2147483647) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(nk + nq + nd + ns));
  LaunchTimer timer(kKidBwdPre, stream);
  if (head_dim == 128)
    hipLaunchKernelGGL(prep_bwd_kernel<128>, grid, dim3(256), 0, stream, a, (int)nk, (int)nq, (int)nd);
  else
    hipLaunchKernelGGL(prep_bwd_kernel<64>, grid, dim3(256), 0, stream, a, (int)nk, (int)nq, (int)nd);
  if (a.kskip != nullptr)
    hipLaunchKernelGGL(key_hull_kernel, dim3((unsigned)(a.B * a.Hkv)), dim3(64), 0, stream, a.kskip, a.Lkp / 64,
                       a.khull);
  return hipGetLastError();
}

// dq = transposed rotation of bf16(acc): the ring's fp32 dq sum cast to the
// input dtype (torch/.../_context_parallel/_attention.py:636) followed by the
// rotation's backward (src/avgen/models/rope.py:332-338 through autograd),
// in one pass.  One thread per 8 channels of a row.
__global__ __launch_bounds__(256) void dq_finish_kernel(const float* __restrict__ acc, int64_t asb, int64_t ash,
                                                        int64_t asl, int H, int L, int D, const float* __restrict__ ct,
                                                        const float* __restrict__ st, int64_t tsb,
                                                        bf16* __restrict__ dq, int64_t dsb, int64_t dsh, int64_t dsl,
                                                        int64_t units) {
  const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= units) return;
  const int cpr = D / 8;
  const int c = (int)(u % cpr);
  const int64_t row = u / cpr;
  const int i = (int)(row % L);
  const int h = (int)((row / L) % H);
  const int b = (int)(row / ((int64_t)L * H));
  const float* ap = acc + b * asb + h * ash + (int64_t)i * asl + 8 * c;
  const f32x4 lo = *reinterpret_cast<const f32x4*>(ap);
  const f32x4 hi = *reinterpret_cast<const f32x4*>(ap + 4);
  u32x4 w = {pack_bf16x2(lo[0], lo[1]), pack_bf16x2(lo[2], lo[3]), pack_bf16x2(hi[0], hi[1]),
             pack_bf16x2(hi[2], hi[3])};
  if (ct) {
    const int64_t t = b * tsb + (int64_t)i * (D / 2) + 4 * c;
    w = rotate8(w, *reinterpret_cast<const f32x4*>(ct + t), *reinterpret_cast<const f32x4*>(st + t), true);
  }
  *reinterpret_cast<u32x4*>(dq + b * dsb + h * dsh + (int64_t)i * dsl + 8 * c) = w;
}

hipError_t launch_dq_finish(const float* acc, int64_t asb, int64_t ash, int64_t asl, int B, int H, int L, int D,
                            const float* cos_t, const float* sin_t, int64_t tsb, bf16* dq, int64_t dsb, int64_t dsh,
                            int64_t dsl, hipStream_t stream) {
  const int64_t units = (int64_t)B * H * L * (D / 8);
  if (units == 0) return hipSuccess;
  const int64_t blocks = (units + 255) / 256;
  if (blocks > 2147483647) return hipErrorInvalidValue;
  LaunchTimer timer(kKidDqFinish, stream);
  hipLaunchKernelGGL(dq_finish_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, acc, asb, ash, asl, H, L, D,
                     cos_t, sin_t, tsb, dq, dsb, dsh, dsl, units);
  return hipGetLastError();
}

}  // namespace avattn
