// gemm_t32.hip -- ternary GEMM on T2 codes with 32x32 int8 MFMA tiles (gfx950),
// for more than 16 activation rows (larger decode batches, prefill). Same
// contract as the reference's gemv_kernel (src/cuda/kernels.cu:238-334).
//
// What bounds it: the vector ALU. Every Q8 block has its own scale, so each
// output takes an int32 -> fp32 conversion and a multiply-add per 32-column
// sub-block; a wave's v_mfma_i32_32x32x32_i8 (one sub-block of 32 weight rows
// x 32 activation rows) comes with 32 such instructions and, measured on
// independent instructions, 110 cycles of a SIMD at 4 waves (118 at 2, 176 at
// one), 21 of them the MFMA's. At gate+up of 512 rows (5120 -> 2 x 17408) the
// kernel holds the vector ALU 94 % of the time (SQ counters) and takes 233 us,
// against 290 for the 16x16x32 tile it replaced, from:
//  - the weights as the MFMA's row operand: a lane's outputs then belong to one
//    activation row, so d is one register per sub-block instead of four, and a
//    lane stores four consecutive outputs at a time;
//  - codes straight from HBM to registers, a block ahead: a lane pair holds a
//    row's 32 bytes of a block, two permlane32 swaps put them in fragment order;
//  - LDS addresses that are a register plus a constant (the loop body is
//    written for both buffers) and weight scales converted when they are
//    staged: 14 additions and 32 mixed-precision multiply-adds a block less
//    (252 -> 233 us);
//  - step e + 1's MFMA and step e + 2's LDS reads issued before step e is scaled.
// The other ways to the float sums cost the same or more: adding 1.5 * 2^23
// through the accumulator and subtracting it (115-128 cycles a step), and
// fp16 MFMA, whose sums are floats already (half the MFMA rate, and q has to
// be converted for every workgroup).
//
// A workgroup is WK groups of WN waves. The groups split the 128-column blocks
// of K (contiguous shares, added in group order at the end); the waves of a
// group share the activation tile (32 MT rows, double-buffered in LDS, one
// barrier a block) and own 32 staged weight rows each (swiglu: 16 gate rows and
// the same 16 up rows). Per output the sums are blk = d * I over a block's
// sub-blocks, then acc = scale * blk + acc per block. For up to 32 rows (one
// activation tile) the epilogue can also write the Q8 of the outputs.
#include <climits>
#include <type_traits>

#include "../../include/btf/hip_abi.h"
#include "common.h"

#pragma clang fp contract(off)

namespace btfhip {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // y rows have any 4-byte alignment

struct T32Args {
  const uint8_t* codes[3];
  const uint16_t* scales[3];
  float* y[3];
  int N[3];
  int ldy[3];
  int tile_start[3];  // first n-tile of each segment; INT_MAX when absent
  const uint8_t* up_codes;
  const uint16_t* up_scales;
  int K, nsub;
  const int8_t* q;
  const float* d;
  int m0, nb;
  int tn, tm;  // tiles along the outputs and the activation rows
  int32_t* dump;
  // optional Q8 of the outputs (segment 0 after the mode), for the next GEMM:
  // q [.][N], d and s [.][N / 32] at activation row m0 + m (one activation tile)
  int8_t* oq;
  float* od;
  int32_t* os;
};

// LDS written by this workgroup visible to it; global loads stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int MT, int WN, int WK, int MODE, bool DUMP>
__global__ void __launch_bounds__(64 * WN * WK, MT == 1 && WN > 1 ? 4 : 3) gemm_t32_kernel(T32Args a) {
  constexpr bool SW = MODE == BTF_GEMV_SWIGLU;
  constexpr int BM = 32 * MT;               // activation rows
  constexpr int TR = SW ? 16 : 32;          // output rows of a 32-row weight tile (swiglu: 16 gate + their 16 up rows)
  constexpr int BNR = TR * WN;              // output rows of the workgroup
  constexpr int TG = 64 * WN;               // threads of a K group
  constexpr int NQ = BM * 8 / TG;           // 16-byte q loads per thread and block
  constexpr int ND = (BM * 4 + TG - 1) / TG;  // d loads per thread and block
  static_assert(BM * 8 % TG == 0, "q loads");
  constexpr int FB = BM * 128;              // q of a block: [row][8 x 16 B], chunk c of row r at slot c ^ (r & 7)
  constexpr int DB = BM * 4 * 4;            // d of a block: [sub-block][row]
  constexpr int SB = WN * 128;              // weight scales of a block: [staged row]
  constexpr int BUF = FB + DB + SB;
  constexpr int RED = WK > 1 ? WK * WN * MT * 4096 : 0;
  constexpr int OUT = MT == 1 ? 32 * (BNR + 1) * 4 : 0;  // outputs to quantize: [activation row][output]
  constexpr int LDS0 = 2 * WK * BUF > RED ? 2 * WK * BUF : RED;
  constexpr int LDS = LDS0 > OUT ? LDS0 : OUT;
  __shared__ __attribute__((aligned(16))) uint8_t lds[LDS];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = w % WN, kg = w / WN;
  const int tg = tid - kg * TG;  // thread within the group
  const int l31 = lane & 31, h = lane >> 5;

  // Workgroup -> tile: consecutive workgroups go to the 8 XCDs in turn, so an
  // XCD takes every eighth weight tile with all its activation tiles: the
  // codes are read into one L2 only.
  const int j = blockIdx.x >> 3;
  const int bx = (j / a.tm) * 8 + (blockIdx.x & 7);
  if (bx >= a.tn) return;
  const int mb = (j % a.tm) * BM;

  const int seg = (bx >= a.tile_start[1]) + (bx >= a.tile_start[2]);
  const uint8_t* codes = seg == 0 ? a.codes[0] : seg == 1 ? a.codes[1] : a.codes[2];
  const uint16_t* scales = seg == 0 ? a.scales[0] : seg == 1 ? a.scales[1] : a.scales[2];
  float* y = seg == 0 ? a.y[0] : seg == 1 ? a.y[1] : a.y[2];
  const int N = seg == 0 ? a.N[0] : seg == 1 ? a.N[1] : a.N[2];
  const int ldy = seg == 0 ? a.ldy[0] : seg == 1 ? a.ldy[1] : a.ldy[2];
  const int tile0 = seg == 0 ? 0 : seg == 1 ? a.tile_start[1] : a.tile_start[2];
  const int K = a.K, nsc = K >> 7, nsub = a.nsub;
  const int n0 = (bx - tile0) * BNR + wn * TR;  // this wave's first output row
  const int k0 = nsc * kg / WK, k1 = nsc * (kg + 1) / WK;
  const int niter = (nsc + WK - 1) / WK;  // the same for every group (barriers)
  uint8_t* buf = lds + kg * 2 * BUF;

  // ---- load sources ----
  const uint8_t* csrc;   // codes: staged row l31, words 4h .. 4h + 3 of a block
  const uint16_t* ssrc;  // scales: staged row l31
  {
    const bool up = SW && l31 >= 16;
    const int nr = n0 + (SW ? (l31 & 15) : l31);
    const int nc = nr < N ? nr : N - 1;
    csrc = (up ? a.up_codes : codes) + (size_t)nc * (K >> 2) + 16 * h;
    ssrc = (up ? a.up_scales : scales) + (size_t)nc * nsc;
  }
  const int8_t* qsrc[NQ];
  uint32_t qdst[NQ];
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    const int e = tg + i * TG, r = e >> 3, c = e & 7;
    const int m = mb + r < a.nb ? mb + r : a.nb - 1;
    qsrc[i] = a.q + (size_t)(a.m0 + m) * K + 16 * c;
    qdst[i] = r * 128 + 16 * (c ^ (r & 7));
  }
  const float* dsrc[ND];
  uint32_t ddst[ND];
#pragma unroll
  for (int i = 0; i < ND; ++i) {
    const int e = tg + i * TG < BM * 4 ? tg + i * TG : BM * 4 - 1;
    const int r = e >> 2, sb = e & 3;
    const int m = mb + r < a.nb ? mb + r : a.nb - 1;
    dsrc[i] = a.d + (size_t)(a.m0 + m) * nsub + sb;
    ddst[i] = FB + (sb * BM + r) * 4;
  }

  u32x4 raw[NQ], cw, cn;
  float rd[ND];
  uint16_t rs;
  auto fetch_act = [&](int kb) {
#pragma unroll
    for (int i = 0; i < NQ; ++i) raw[i] = *reinterpret_cast<const u32x4*>(qsrc[i] + (size_t)kb * 128);
#pragma unroll
    for (int i = 0; i < ND; ++i) rd[i] = dsrc[i][4 * (size_t)kb];
    rs = ssrc[kb];
  };
  auto fetch_codes = [&](int kb) { cn = *reinterpret_cast<const u32x4*>(csrc + (size_t)kb * 32); };
  auto stage = [&](int b) {  // (b is a constant at each call: the LDS addresses below are registers plus constants)
    uint8_t* o = buf + b * BUF;
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      *reinterpret_cast<u32x4*>(o + qdst[i]) = raw[i];
    }
#pragma unroll
    for (int i = 0; i < ND; ++i) *reinterpret_cast<float*>(o + ddst[i]) = rd[i];
    *reinterpret_cast<float*>(o + FB + DB + (wn * 32 + l31) * 4) = h2f(rs);  // (both halves: the same value)
  };

  f16v acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][r] = 0.f;
  v16i zero;
#pragma unroll
  for (int r = 0; r < 16; ++r) zero[r] = 0;

  if (k0 < k1) {
    fetch_act(k0);
    fetch_codes(k0);
    stage(0);
    cw = cn;
    if (k0 + 1 < k1) {
      fetch_act(k0 + 1);
      fetch_codes(k0 + 1);
    }
  }
  lds_barrier();
  const uint32_t arow = l31 * 128;
  uint32_t aoff[4];  // this lane's q chunk of sub-block s (rows of the other activation tiles: + 4096 each)
#pragma unroll
  for (int s = 0; s < 4; ++s) aoff[s] = arow + 16 * ((2 * s + h) ^ (l31 & 7));
  auto block = [&](int it, auto bufi) {
    constexpr int B = decltype(bufi)::value;
    const int kb = k0 + it;
    if (kb < k1) {
      const uint8_t* b = buf + B * BUF;
      // words of sub-block s in lane group h: 2s + h (the load gave group h words 4h .. 4h + 3)
      const auto r01 = __builtin_amdgcn_permlane32_swap(cw.x, cw.y, false, false);
      const auto r23 = __builtin_amdgcn_permlane32_swap(cw.z, cw.w, false, false);
      const uint32_t word[4] = {r01[0], r23[0], r01[1], r23[1]};
      cw = cn;
      v4i wf[4];
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int k = 0; k < 4; ++k)  // codes 0 / 1 / 2 -> int8 -1 / 0 / +1
          wf[s][k] = (int)__builtin_amdgcn_perm(0u, 0x000100FFu, (word[s] >> (2 * k)) & 0x03030303u);
      // the next block's activation goes to the other buffer: its loads were issued a block ago
      if (kb + 1 < k1) {
        stage(B ^ 1);
        if (kb + 2 < k1) {
          fetch_act(kb + 2);
          fetch_codes(kb + 2);
        }
      }
      // Steps e = (activation tile i, sub-block s). Step e + 1's MFMA and step
      // e + 2's LDS reads are issued before step e is scaled, so that the
      // matrix core and the LDS run under the vector ALU's work of this wave.
      constexpr int E = 4 * MT;
      v4i af[2];
      float dv[3];
      v16i I[2];
      auto rd_act = [&](int e) {
        const int i = e >> 2, s = e & 3;
        af[e & 1] = *reinterpret_cast<const v4i*>(b + aoff[s] + 4096 * i);
        dv[e % 3] = *reinterpret_cast<const float*>(b + FB + (s * BM + 32 * i + l31) * 4);
      };
      auto mma = [&](int e) { I[e & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf[e & 3], af[e & 1], zero, 0, 0, 0); };
      rd_act(0);
      rd_act(1);
      mma(0);
      float sc[16];
      f16v blk;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        if (!DUMP && e == 2) {
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const f32x4 sv = *reinterpret_cast<const f32x4*>(b + FB + DB + (wn * 32 + 8 * c + 4 * h) * 4);
#pragma unroll
            for (int r = 0; r < 4; ++r) sc[4 * c + r] = sv[r];
          }
        }
        const int i = e >> 2, s = e & 3;
        if (e + 1 < E) mma(e + 1);
        if (e + 2 < E) rd_act(e + 2);
        const float d = dv[e % 3];
        if constexpr (DUMP) {  // the exact I of every (row, output, sub-block)
          const int m = mb + 32 * i + l31;
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int n = n0 + 8 * (r >> 2) + 4 * h + (r & 3);
            if (m < a.nb && n < N) a.dump[((size_t)(a.m0 + m) * N + n) * nsub + kb * 4 + s] = I[e & 1][r];
          }
        } else {
#pragma unroll
          for (int r = 0; r < 16; ++r)
            blk[r] = s == 0 ? d * (float)I[e & 1][r] : fmaf(d, (float)I[e & 1][r], blk[r]);
          if (s == 3) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][r] = fmaf(sc[r], blk[r], acc[i][r]);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    lds_barrier();
  };
  for (int it = 0; it < niter; it += 2) {
    block(it, std::integral_constant<int, 0>{});
    if (it + 1 < niter) block(it + 1, std::integral_constant<int, 1>{});
  }
  if constexpr (DUMP) return;

  // ---- epilogue: lane holds activation row mb + 32 i + l31; register r its staged row
  // 8 (r / 4) + 4 h + r % 4 (swiglu: gate rows in registers 0-7, their up rows in 8-15),
  // so four registers (a chunk c) are four consecutive outputs ----
  const bool quant = MT == 1 && a.oq;  // (uniform)
  auto emit = [&](int i, int c, const f32x4& g, const f32x4& u) {
    const int m = mb + 32 * i + l31;
    const bool live = m < a.nb;
    float* yr = y + (size_t)(a.m0 + (live ? m : 0)) * ldy;
    const int n = n0 + 8 * c + 4 * h;
    f32x4u v;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if constexpr (SW)
        v[r] = g[r] / (1.0f + expf(-g[r])) * u[r];
      else
        v[r] = g[r];
    }
    if (live && n + 3 < N) {
      f32x4u* o = reinterpret_cast<f32x4u*>(yr + n);
      if constexpr (MODE == BTF_GEMV_ADD) {
        const f32x4u old = *o;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = old[r] + v[r];
      }
      *o = v;
    } else if (live) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n + r < N) yr[n + r] = MODE == BTF_GEMV_ADD ? yr[n + r] + v[r] : v[r];
    }
    if (quant) {  // (N % 32 == 0: live blocks are whole)
      float* ol = reinterpret_cast<float*>(lds) + l31 * (BNR + 1) + wn * TR + 8 * c + 4 * h;
#pragma unroll
      for (int r = 0; r < 4; ++r) ol[r] = v[r];
    }
  };
  constexpr int NC = SW ? 2 : 4;  // chunks of outputs
  auto chunk = [&](int i, int c) { return f32x4{acc[i][4 * c], acc[i][4 * c + 1], acc[i][4 * c + 2], acc[i][4 * c + 3]}; };
  if constexpr (WK > 1) {
    // The groups' partial sums, added in group order: group c adds and writes
    // chunk c, so a lane reads WK 16-byte words (swiglu: twice that) in a row
    // and not, as one group adding them all would, 16 (WK - 1) registers.
    static_assert(WK >= NC, "a group per chunk");
    f32x4* red = reinterpret_cast<f32x4*>(lds);  // [kg][wn][tile][chunk][lane] (over the buffers: all reads are done)
    auto slot = [&](int g, int i, int c) { return (((g * WN + wn) * MT + i) * 4 + c) * 64 + lane; };
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c) red[slot(kg, i, c)] = chunk(i, c);
    lds_barrier();
    f32x4 g[MT], u[MT];
    if (kg < NC) {
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        g[i] = red[slot(0, i, kg)];
        if constexpr (SW) u[i] = red[slot(0, i, kg + 2)];
#pragma unroll
        for (int k = 1; k < WK; ++k) {
          const f32x4 gk = red[slot(k, i, kg)];
#pragma unroll
          for (int r = 0; r < 4; ++r) g[i][r] = g[i][r] + gk[r];
          if constexpr (SW) {
            const f32x4 uk = red[slot(k, i, kg + 2)];
#pragma unroll
            for (int r = 0; r < 4; ++r) u[i][r] = u[i][r] + uk[r];
          }
        }
      }
    }
    if (quant) lds_barrier();  // every read of the partial sums is done
    if (kg < NC) {
#pragma unroll
      for (int i = 0; i < MT; ++i) emit(i, kg, g[i], u[i]);
    }
  } else {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int c = 0; c < NC; ++c) emit(i, c, chunk(i, c), SW ? chunk(i, c + 2) : f32x4{});
  }
  if constexpr (MT == 1) {
    if (quant) {
      lds_barrier();
      // a half-wave per (activation row, 32-output block), with the q8 kernel's arithmetic
      const int b0 = (bx - tile0) * (BNR / 32), nblk = N / 32;
      for (int e = 2 * w + h; e < 32 * (BNR / 32); e += 2 * WN * WK) {
        const int mm = e & 31, bl = e >> 5;
        float dq;
        int sq;
        const int q = q8_half(reinterpret_cast<const float*>(lds)[mm * (BNR + 1) + 32 * bl + l31], dq, sq);
        uint32_t wq = (uint32_t)(q & 0xff) << (8 * (l31 & 3));
        wq |= (uint32_t)dpp_i<0xB1>((int)wq);  // quad_perm(1,0,3,2)
        wq |= (uint32_t)dpp_i<0x4E>((int)wq);  // quad_perm(2,3,0,1)
        if (mb + mm < a.nb && b0 + bl < nblk) {
          const size_t mr = (size_t)(a.m0 + mb + mm);
          if ((l31 & 3) == 0) *reinterpret_cast<uint32_t*>(a.oq + mr * N + 32 * (b0 + bl) + l31) = wq;
          if (l31 == 0) {
            a.od[mr * nblk + b0 + bl] = dq;
            a.os[mr * nblk + b0 + bl] = sq;
          }
        }
      }
    }
  }
}

template <int MT, int WN, int WK>
void by_mode(int mode, const T32Args& a, int grid, hipStream_t st) {  // (a by reference: the grid's computation sets it)
  const dim3 blk(64 * WN * WK);
  if (a.dump)
    hipLaunchKernelGGL((gemm_t32_kernel<MT, WN, WK, BTF_GEMV_STORE, true>), dim3(grid), blk, 0, st, a);
  else if (mode == BTF_GEMV_STORE)
    hipLaunchKernelGGL((gemm_t32_kernel<MT, WN, WK, BTF_GEMV_STORE, false>), dim3(grid), blk, 0, st, a);
  else if (mode == BTF_GEMV_ADD)
    hipLaunchKernelGGL((gemm_t32_kernel<MT, WN, WK, BTF_GEMV_ADD, false>), dim3(grid), blk, 0, st, a);
  else
    hipLaunchKernelGGL((gemm_t32_kernel<MT, WN, WK, BTF_GEMV_SWIGLU, false>), dim3(grid), blk, 0, st, a);
}

}  // namespace

int gemm_t32(const GemvSeg* segs, int nseg, int K, int m0, int nb, const Q8& act, int mode, int32_t* dump,
             hipStream_t st, const Q8* qout) {
  T32Args a{};
  const int nuse = mode == BTF_GEMV_SWIGLU ? 1 : nseg;
  a.K = K;
  a.nsub = K / 32;
  a.q = act.q;
  a.d = act.d;
  a.m0 = m0;
  a.nb = nb;
  a.dump = dump;
  if (mode == BTF_GEMV_SWIGLU) {
    a.up_codes = segs[1].codes;
    a.up_scales = segs[1].scales;
  }
  if (qout) {
    a.oq = const_cast<int8_t*>(qout->q);  // (Q8 holds read-only views; this one is written)
    a.od = const_cast<float*>(qout->d);
    a.os = const_cast<int32_t*>(qout->s);
  }
  // sets the n-tiles of `rows` output rows and the m-tiles of bm rows; returns the grid, which
  // covers 8 n-tiles at a time (see the kernel's mapping)
  auto tiles = [&](int rows, int bm) {
    int t = 0;
    for (int i = 0; i < 3; ++i) {
      if (i < nuse) {
        a.codes[i] = segs[i].codes;
        a.scales[i] = segs[i].scales;
        a.y[i] = segs[i].y;
        a.N[i] = segs[i].N;
        a.ldy[i] = segs[i].ldy;
        a.tile_start[i] = t;
        t += (segs[i].N + rows - 1) / rows;
      } else {
        a.tile_start[i] = INT_MAX;
      }
    }
    a.tn = t;
    a.tm = (nb + bm - 1) / bm;
    return (t + 7) / 8 * 8 * a.tm;
  };
  // Tile by the number of 32 x 32 output tiles (waves' worth of work; the chip
  // holds 4096 waves at 4 per SIMD). Many: 64 activation rows per wave halve
  // the decode per output, K unsplit. Fewer: 32 rows, and K split over the
  // groups of a workgroup so that every SIMD has waves to overlap. Measured
  // (us, tiles; the chosen one first): gate+up 5120 -> 2 x 17408, 512 rows
  // (17408 tiles) 2,4,1 233, 1,4,1 259, 1,2,4 300; 128 rows (4352) 1,4,1 82,
  // 2,4,1 84, 1,2,4 81; 64 rows (2176) 1,2,4 48, 1,4,1 51, 1,2,8 63; down
  // 17408 -> 5120, 203 rows (1120) 1,2,4 93, 1,4,1 117, 1,2,8 103; 5120 ->
  // 5120, 64 rows (320) 1,2,8 13.4, 1,2,4 14.0, 1,1,4 15.6; gate+up of 32 rows
  // (1088) 1,2,4 34, 1,4,1 37, 1,2,8 41; 5120 -> 3 x 5120, 32 rows (480)
  // 1,2,8 15.8, 1,2,4 16.2; 2048 -> 2 x 2048, 96 rows (384) 1,2,4 7.7, 1,2,8
  // 8.7. At most one tile per CU: a workgroup of one tile, on as many CUs as
  // there are tiles; 32 rows, 5120 -> 5120 (160) 1,1,8 9.7, 1,2,8 12.8, 1,1,4
  // 11.4; down (160) 1,1,12 27.4, 1,1,8 28.8, 1,2,8 36; 4096 -> 2048 (64) 1,1,8
  // 7.8, 1,1,12 8.1, 1,2,8 10.5; 1024 -> 1024 (32) 1,1,4 4.22, 1,1,8 4.22, 1,2,8
  // 5.4; one block per group: 512 -> 3 x 4096, 64 rows (768) 1,1,4 5.0, 1,2,4 5.5.
  // K unsplit from 3000 tiles: 3072 -> 3072, 1000 rows (3072) 1,4,1 37, 1,2,4 40;
  // and from 1024 where a group would have at most one block: 256 -> 3 x 2048,
  // 512 rows (3072) 1,4,1 7.2, 1,2,4 12.4.
  // (qout does not change the K split: y is the same with and without it.)
  const int per = mode == BTF_GEMV_SWIGLU ? 16 : 32;  // output rows of a wave
  tiles(per, 32);
  const int64_t t32 = (int64_t)a.tn * a.tm;
  if (t32 == 0) return BTF_OK;
  if (t32 >= 8192 && nb > 32) {
    by_mode<2, 4, 1>(mode, a, tiles(4 * per, 64), st);
  } else if (t32 >= 3000 || (K <= 512 && t32 >= 1024)) {
    by_mode<1, 4, 1>(mode, a, tiles(4 * per, 32), st);
  } else if (t32 <= 256 || (K <= 512 && t32 < 1024)) {
    // (a swiglu's Q8 blocks are two waves wide: the same K split, so the same y)
    const bool wide = qout && mode == BTF_GEMV_SWIGLU;
    if (K <= 1024) {
      if (wide) by_mode<1, 2, 4>(mode, a, tiles(2 * per, 32), st);
      else by_mode<1, 1, 4>(mode, a, tiles(per, 32), st);
    } else if (K < 12288 || mode == BTF_GEMV_SWIGLU) {
      if (wide) by_mode<1, 2, 8>(mode, a, tiles(2 * per, 32), st);
      else by_mode<1, 1, 8>(mode, a, tiles(per, 32), st);
    } else {
      by_mode<1, 1, 12>(mode, a, tiles(per, 32), st);
    }
  } else if (t32 >= 500 || K < 4096) {
    by_mode<1, 2, 4>(mode, a, tiles(2 * per, 32), st);
  } else {
    by_mode<1, 2, 8>(mode, a, tiles(2 * per, 32), st);
  }
  return launch_status("gemm_t32_kernel");
}

}  // namespace btfhip
