// prep.hip -- activation prep for the ternary matmul (gfx950).
//
// Behaviour of the reference's launch_prep (src/cuda/kernels.cuh:40-43) and
// of its CPU twin EmuDecoder::prep (src/emu_decoder.cpp:122-140) with
// bd::rmsnorm and bd::hadamard_input (ref/bonsai-decoder/src/cpu_ops.cpp:
// 90-127):
//   x [M][ldx] -> [RMSNorm * w] -> tiled->grouped perm -> signs ->
//   blockwise WHT (x 1/sqrt(block)) -> Q8_0 (q, d, s) per 32 values.
// As on the CPU, the perm and the signs belong to the transform: with
// block == 0 neither is applied.
//
// Three kernels:
//  * q8_kernel: no norm and no transform (every quantize feeding a GEMV in the
//    synthetic workloads). Four lanes own one 32-value block, 8 values each;
//    amax and sum(q) are 2-step DPP quad reductions. Bit-exact with
//    include/btf/packed.hpp:117-134: d = fp16_rn(amax/127) (IEEE division),
//    q = rint(x * (127/amax)) with ties to even, s = sum q. An all-zero block
//    gets d = +-0 with the sign of its last element, as the CPU loop does.
//  * prep_quad_kernel<NORM, PERM, VEC>: the full transform, four waves per
//    (1024-value slice, row): the FWHT runs in the CPU's stage order, so
//    without the norm the result is bit-exact; the RMSNorm's double sum of
//    squares is taken in a fixed canonical order (per 32-value block, then over
//    the blocks), so its last bit can differ from the CPU's sequential sum (the
//    reference's own GPU kernel differs likewise);
//  * prep_slice_kernel<VEC>: the same transform on one wave per slice
//    (slice.h), for prompt-sized calls without norm and gather.
#include <cmath>

#include "../../include/btf/hip_abi.h"
#include "common.h"
#include "slice.h"

#pragma clang fp contract(off)

namespace btfhip {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Quantize 8 consecutive values of one Q8 block held by this lane; the 4
// lanes of a DPP quad hold the block. Returns the two packed q words; d and s
// are valid in every lane of the quad.
__device__ __forceinline__ void q8_quad(const float (&v)[8], uint32_t& q0, uint32_t& q1, float& d, int& s) {
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(v[i]));
  amax = quad_max_f(amax);
  // sign of the block's last value, for the all-zero case
  const float last = dpp_f<0xFF>(v[7]);  // quad_perm(3,3,3,3)
  float dd = h2f(f2h_bits(amax / 127.0f));
  if (amax == 0.f) dd = copysignf(0.f, last);
  d = dd;
  const float id = amax != 0.f ? 127.0f / amax : 0.f;
  int qi[8];
  int sum = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    qi[i] = (int)__builtin_rintf(v[i] * id);
    sum += qi[i];
  }
  q0 = (uint32_t)(qi[0] & 0xff) | ((uint32_t)(qi[1] & 0xff) << 8) | ((uint32_t)(qi[2] & 0xff) << 16) |
       ((uint32_t)(qi[3] & 0xff) << 24);
  q1 = (uint32_t)(qi[4] & 0xff) | ((uint32_t)(qi[5] & 0xff) << 8) | ((uint32_t)(qi[6] & 0xff) << 16) |
       ((uint32_t)(qi[7] & 0xff) << 24);
  s = quad_sum_i(sum);
}

// One lane per 8 values. Grid covers M * n / 8 lanes exactly (multiple of 4).
template <bool VEC>
__global__ void __launch_bounds__(256) q8_kernel(const float* __restrict__ x, int ldx, int n, int64_t total_lanes,
                                                  int8_t* __restrict__ q, float* __restrict__ d,
                                                  int32_t* __restrict__ s) {
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  // Out-of-range lanes still run the quad reductions (on zeros) but store nothing.
  const bool live = gid < total_lanes;
  const int64_t g = live ? gid : 0;
  const int lanes_per_row = n >> 3;
  const int64_t m = g / lanes_per_row;
  const int c8 = (int)(g - m * lanes_per_row);  // 8-value chunk within the row
  const float* xp = x + m * (int64_t)ldx + 8 * c8;
  float v[8];
  if (VEC) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(xp);
    const f32x4 b = *reinterpret_cast<const f32x4*>(xp + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = xp[i];
  }
  uint32_t q0, q1;
  float dd;
  int ss;
  q8_quad(v, q0, q1, dd, ss);
  if (!live) return;
  uint32_t* qp = reinterpret_cast<uint32_t*>(q + m * (int64_t)n + 8 * c8);
  qp[0] = q0;
  qp[1] = q1;
  if ((c8 & 3) == 0) {
    const int64_t bi = m * (int64_t)(n >> 5) + (c8 >> 2);
    d[bi] = dd;
    s[bi] = ss;
  }
}

// ---- full prep ----
// One workgroup of four waves per (1024-value slice, row), every one
// independent; thread t holds values 4 t .. 4 t + 3 of the slice. With the
// norm, the workgroup first forms the row's RMSNorm scale itself: the
// canonical sums of squares of the row's 32-value blocks (eight lanes each,
// the pairwise tree over the value index bits) go to LDS, lane l of every wave
// adds blocks l, l + 64, ... in order, then the wave sum (slice.h) -- the order
// in which the step program sums its producers' block sums, so both get the
// same scale bit for bit. Then the slice: gather through the perm,
// (x * scale) * w, the normed values to xn_out, * signs, the blockwise FWHT
// (stages len 1 and 2 in a lane, 4 .. 128 across lanes, 256 and 512 across
// waves through LDS in one exchange), * 1/sqrt(block), the Q8 of each
// eight-lane block.
// What bounds it: at decode sizes the latency of one wave's chain (with one
// wave of 16 values a lane it issued 4x the dependent instructions, alone on its
// SIMD), with the norm at prompt sizes the row's sums that every slice forms
// (read in whole lines here, 128 bytes a lane before). Measured per launch in a
// graph of them, one wave per slice -> four (us): 8 rows of 5120 with norm 4.2
// -> 3.4, 8 rows of 17408 without 2.8 -> 2.4, with the gather 4.3 -> 2.9; 512
// rows of 5120 with norm 12.9 -> 11.5, of 17408 76.8 -> 53.8.
struct PrepArgs {
  const float* x;
  int ldx, n;
  const float* normw;
  float eps;
  int block, hd, nk, rep;  // rep > 1: tiled -> grouped gather
  float hs;                // 1/sqrtf(block) (block > 0)
  const float* signs;
  float* xn;
  int ldxn;
  int8_t* q;
  float* d;
  int32_t* s;
};

// 16 consecutive values of row xr from index c0 (16-byte loads when VEC).
template <bool VEC>
__device__ __forceinline__ void load16(const float* xr, int c0, float (&v)[16]) {
  if (VEC) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const f32x4 t = reinterpret_cast<const f32x4*>(xr + c0)[k];
      v[4 * k] = t.x;
      v[4 * k + 1] = t.y;
      v[4 * k + 2] = t.z;
      v[4 * k + 3] = t.w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = xr[c0 + i];
  }
}

// Prompt sizes without norm and gather: one wave per slice, 16 values a lane. The Q8's
// divisions and the addressing are paid once per 16 values instead of once per 4, which
// counts when every SIMD has waves (512 rows of 17408: 11.1 us against 13.3 with four
// waves per slice; 64 rows of 5120, where latency counts: 2.9 against 2.6).
template <bool VEC>
__global__ void __launch_bounds__(64) prep_slice_kernel(PrepArgs a) {
  const int lane = threadIdx.x, m = blockIdx.y;
  const float* xr = a.x + (size_t)m * a.ldx;
  const int c0 = blockIdx.x * kSliceVals + 16 * lane;
  const bool live = c0 < a.n;  // a.n % 32 == 0: a lane pair is all in or all out
  float v[16];
  if (live) {
    load16<VEC>(xr, c0, v);
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = 0.f;
  }
  if (a.xn && live) {
    float* xo = a.xn + (size_t)m * a.ldxn + c0;
#pragma unroll
    for (int i = 0; i < 16; ++i) xo[i] = v[i];
  }
  if (a.block > 0) {
    if (a.signs && live)
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = v[i] * a.signs[c0 + i];
    slice_fwht(v, lane, a.block);
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = v[i] * a.hs;
  }
  uint32_t qw[4];
  float dd;
  int ss;
  q8_pair(v, qw, dd, ss);
  if (live) {
    uint32_t* qp = reinterpret_cast<uint32_t*>(a.q + (size_t)m * a.n + c0);
    qp[0] = qw[0];
    qp[1] = qw[1];
    qp[2] = qw[2];
    qp[3] = qw[3];
    if (!(lane & 1)) {
      const size_t bi = (size_t)m * (a.n >> 5) + (c0 >> 5);
      a.d[bi] = dd;
      a.s[bi] = ss;
    }
  }
}

// 4 consecutive values of row xr from index c0 (a 16-byte load when VEC).
template <bool VEC>
__device__ __forceinline__ void load4(const float* xr, int c0, float (&v)[4]) {
  if (VEC) {
    const f32x4 t = *reinterpret_cast<const f32x4*>(xr + c0);
    v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = xr[c0 + i];
  }
}

constexpr int kPrepThreads = kSliceVals / 4;
constexpr int kNormBlocks = 1024;  // block sums held in LDS at a time

template <bool NORM, bool PERM, bool VEC>
__global__ void __launch_bounds__(kPrepThreads) prep_quad_kernel(PrepArgs a) {
  __shared__ f32x4 xch[kPrepThreads];
  __shared__ double bs[NORM ? kNormBlocks : 1];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, m = blockIdx.y;
  const float* xr = a.x + (size_t)m * a.ldx;
  const int c0 = blockIdx.x * kSliceVals + 4 * tid;
  const bool live = c0 < a.n;  // a.n % 32 == 0: an eight-lane block is all in or all out
  // the slice and its factors, in flight under the norm's sums
  float v[4] = {0.f, 0.f, 0.f, 0.f}, nw[4] = {0.f, 0.f, 0.f, 0.f}, sg[4] = {1.f, 1.f, 1.f, 1.f};
  if (live) {
    if (PERM) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int src = perm_src(c0 + i, a.hd, a.nk, a.rep);
        v[i] = xr[src];
        if (NORM) nw[i] = a.normw[src];
      }
    } else {
      load4<VEC>(xr, c0, v);
      if (NORM) load4<false>(a.normw, c0, nw);
    }
    if (a.signs) load4<false>(a.signs, c0, sg);
  }
  float scale = 1.0f;
  if (NORM) {
    double acc = 0.0;
    const int nblk = a.n >> 5;
    for (int b0 = 0; b0 < nblk; b0 += kNormBlocks) {
      const int cend = 32 * (b0 + kNormBlocks) < a.n ? 32 * (b0 + kNormBlocks) : a.n;
      if (b0) __syncthreads();  // the sums before are read
      constexpr int U = 5;      // passes of 1024 values with their loads in flight together
      for (int cb = 32 * b0; cb < cend; cb += U * kSliceVals) {
        float t[U][4];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int c = cb + u * kSliceVals + 4 * tid;
          load4<VEC>(xr, c < cend ? c : 4 * (tid & 7), t[u]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int c = cb + u * kSliceVals + 4 * tid;
          double s[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) s[i] = (double)t[u][i] * (double)t[u][i];
          double sum = (s[0] + s[1]) + (s[2] + s[3]);
          sum = sum + lane_xor_d<1>(sum);
          sum = sum + lane_xor_d<2>(sum);
          sum = sum + lane_xor_d<4>(sum);
          if (c < cend && (lane & 7) == 0) bs[(c >> 5) - b0] = sum;
        }
      }
      __syncthreads();
      const int nb = nblk - b0 < kNormBlocks ? nblk - b0 : kNormBlocks;
      for (int b = lane; b < nb; b += 64) acc += bs[b];
    }
    scale = norm_scale_of(acc, a.n, a.eps);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (v[i] * scale) * nw[i];
  }
  if (a.xn && live) {
    float* xo = a.xn + (size_t)m * a.ldxn + c0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float u = xr[c0 + i];
      if (NORM) u = (u * scale) * a.normw[c0 + i];
      xo[i] = u;
    }
  }
  if (a.block > 0) {
    if (a.signs)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = v[i] * sg[i];
    if (a.block > 1) istage<1>(v);
    if (a.block > 2) istage<2>(v);
    if (a.block > 4) xstage<1>(v, lane);
    if (a.block > 8) xstage<2>(v, lane);
    if (a.block > 16) xstage<4>(v, lane);
    if (a.block > 32) xstage<8>(v, lane);
    if (a.block > 64) xstage<16>(v, lane);
    if (a.block > 128) xstage<32>(v, lane);
    if (a.block > 256) {  // waves w and w ^ 1, then pairs of them
      xch[tid] = f32x4{v[0], v[1], v[2], v[3]};
      __syncthreads();
      const f32x4 p = xch[tid ^ 64];
      const bool up1 = w & 1, up2 = w & 2;
      if (a.block > 512) {
        const f32x4 o = xch[tid ^ 128], po = xch[tid ^ 192];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float t = up1 ? p[i] - v[i] : v[i] + p[i];
          const float to = up1 ? po[i] - o[i] : o[i] + po[i];
          v[i] = up2 ? to - t : t + to;
        }
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = up1 ? p[i] - v[i] : v[i] + p[i];
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = v[i] * a.hs;
  }
  float dd;
  int ss;
  const uint32_t qw = q8_oct(v, dd, ss);
  if (live) {
    *reinterpret_cast<uint32_t*>(a.q + (size_t)m * a.n + c0) = qw;
    if ((lane & 7) == 0) {
      const size_t bi = (size_t)m * (a.n >> 5) + (c0 >> 5);
      a.d[bi] = dd;
      a.s[bi] = ss;
    }
  }
}

}  // namespace

int prep(const float* x, int ldx, int M, int n, const float* normw, float eps, int block, int perm_hd, int perm_nk,
         int perm_rep, const float* signs, float* xn_out, int ldxn, int8_t* q, float* d, int32_t* s, hipStream_t st,
         const DevState& ds) {
  (void)ds;
  if (!normw && block <= 0 && !xn_out) {
    const int64_t lanes = (int64_t)M * (n / 8);
    const int64_t grid = (lanes + 255) / 256;
    const bool vec = ((reinterpret_cast<uintptr_t>(x) & 15) == 0) && (ldx % 4 == 0);
    if (vec)
      hipLaunchKernelGGL(q8_kernel<true>, dim3((unsigned)grid), dim3(256), 0, st, x, ldx, n, lanes, q, d, s);
    else
      hipLaunchKernelGGL(q8_kernel<false>, dim3((unsigned)grid), dim3(256), 0, st, x, ldx, n, lanes, q, d, s);
    return launch_status("q8_kernel");
  }
  // The transform acts in blocks of `block` values (a power of two) that
  // must divide the span: the largest power of two <= 1024 dividing n.
  int span = 1024;
  while (n % span) span >>= 1;
  if (block > 0 && span % block) return fail(BTF_ERR_ARGS, "prep: hadamard block does not divide the span");
  PrepArgs p{};
  p.x = x;
  p.ldx = ldx;
  p.n = n;
  p.normw = normw;
  p.eps = eps;
  p.block = block > 0 ? block : 0;
  const bool perm = block > 0 && perm_rep > 1;
  p.hd = perm_hd;
  p.nk = perm_nk;
  p.rep = perm_rep;
  p.hs = block > 0 ? 1.0f / std::sqrt((float)block) : 1.0f;
  p.signs = block > 0 ? signs : nullptr;
  p.xn = xn_out;
  p.ldxn = ldxn;
  p.q = q;
  p.d = d;
  p.s = s;
  const bool vec = ((reinterpret_cast<uintptr_t>(x) & 15) == 0) && (ldx % 4 == 0);
  const dim3 grid((n + kSliceVals - 1) / kSliceVals, M);
  // prompt-sized calls without norm and gather: see prep_slice_kernel (the two
  // cross at about 1200 slices: 256 rows of 5120 3.80 against 3.75, 128 rows
  // of 17408 4.7 against 5.1)
  if (!normw && !perm && (int64_t)grid.x * M > 1280) {
    if (vec)
      hipLaunchKernelGGL(prep_slice_kernel<true>, grid, dim3(64), 0, st, p);
    else
      hipLaunchKernelGGL(prep_slice_kernel<false>, grid, dim3(64), 0, st, p);
    return launch_status("prep_slice_kernel");
  }
#define BTF_PREP_LAUNCH(NORM, PERM, VEC) \
  hipLaunchKernelGGL((prep_quad_kernel<NORM, PERM, VEC>), grid, dim3(kPrepThreads), 0, st, p)
  if (normw) {
    if (perm) {
      if (vec) BTF_PREP_LAUNCH(true, true, true); else BTF_PREP_LAUNCH(true, true, false);
    } else {
      if (vec) BTF_PREP_LAUNCH(true, false, true); else BTF_PREP_LAUNCH(true, false, false);
    }
  } else {
    if (perm) {
      if (vec) BTF_PREP_LAUNCH(false, true, true); else BTF_PREP_LAUNCH(false, true, false);
    } else {
      if (vec) BTF_PREP_LAUNCH(false, false, true); else BTF_PREP_LAUNCH(false, false, false);
    }
  }
#undef BTF_PREP_LAUNCH
  return launch_status("prep_quad_kernel");
}

}  // namespace btfhip
