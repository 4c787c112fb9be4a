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
// kernel holds the vector ALU 93 % of the time (SQ counters) and takes 240 us,
// against 280 for the 16x16x32 tile it replaced, from:
//  - the weights as the MFMA's row operand: a lane's outputs then belong to one
//    activation row, so d is one register per sub-block instead of four, and a
//    lane stores four consecutive outputs at a time;
//  - codes straight from HBM to registers, a block ahead: a lane pair holds a
//    row's 32 bytes of a block, two permlane32 swaps put them in fragment order;
//  - LDS addresses that are a register plus a constant (the loop body is
//    written for both buffers) and weight scales converted when they are
//    staged: 14 additions and 32 mixed-precision multiply-adds a block less
//    (252 -> 233 us, K in one sum);
//  - step e + 1's MFMA and step e + 2's LDS reads issued before step e is scaled.
// The other ways to the float sums cost the same or more: adding 1.5 * 2^23
// through the accumulator and subtracting it (115-128 cycles a step), and
// fp16 MFMA, whose sums are floats already (half the MFMA rate, and q has to
// be converted for every workgroup).
//
// A workgroup is WK groups of WN waves. The groups split the 128-column blocks
// of K (contiguous parts, added in order at the end); the waves of a
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

// The order of the sums. K is cut into G contiguous shares of its 128-column
// blocks: share g is blocks nsc g / G .. nsc (g + 1) / G, summed in order from
// zero, and the shares are added in order. G follows from the matrix alone and
// every tile shape keeps to it, so an output of more than 16 rows has the same
// bits whatever the launch's rows, segments and mode are. A tile that splits K
// over fewer groups than G sets the sums of each share aside in LDS.
// G is 8 from K = 4096, where a launch of few rows splits K over 8 groups of waves
// (32 rows of 5120 -> 5120: 9.5 us, over 4 groups 11.2; 3072 -> 3072 6.6 / 7.5). 4
// below: eight chains of fewer than four blocks and their adds are further off 64
// bits than four (2304 -> 6000: 6.4e-8 against 5.9e-8; even at 4096). And 4 for
// 16384 outputs and more, which fill the chip by themselves: a tile that does not
// split K pays for each share (gate+up of 512 rows, 5120 -> 2 x 17408: 238 us with
// all of K in one sum, 244 in 4 shares, 249 in 8; 2048 -> 2 x 8192, 512 rows, 49.5,
// 52.6, 55.3).
__host__ __device__ constexpr int k_shares_log2(int nsc, int N) { return nsc < 32 || N >= 16384 ? 2 : 3; }

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

// MS: the most shares of K that a group holds (1: exactly one, so nothing is set aside).
template <int MT, int WN, int WK, int MS, int MODE, bool DUMP>
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
  constexpr int PART = WN * MT * 4096;      // a group's sums: [tile, chunk][thread]
  constexpr int SAVE = MS > 1 ? PART : 0;  // those of the shares before its last one
  constexpr int GRP = 2 * BUF + SAVE;       // LDS of a group
  constexpr int OUT = MT == 1 ? 32 * (BNR + 1) * 4 : 0;  // outputs to quantize: [activation row][output]
  constexpr int LDS = WK * GRP > OUT ? WK * GRP : OUT;
  static_assert(WK == 1 || PART <= 2 * BUF, "the partial sums go over the buffers");
  __shared__ __attribute__((aligned(16))) uint8_t lds[LDS];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = w % WN, kg = WK == 1 ? 0 : w / WN;
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
  uint8_t* buf = lds + kg * GRP;

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
  // This thread's 16-byte slot for chunk c of activation tile i in a part of PART bytes. Its
  // offset takes no register of the loop: one group has it in its first q offset, more
  // compute it anew from the thread id (a value the compiler keeps spills in <1,2,4>).
  auto slot = [&](uint8_t* part, int i, int c) -> f32x4& {
    int off;
    if constexpr (WK == 1) {
      off = (int)qdst[0];
    } else {
      int t = threadIdx.x;
      asm volatile("" : "+v"(t));
      off = 16 * (t - kg * TG);
    }
    return *reinterpret_cast<f32x4*>(part + off + (4 * i + c) * 16 * TG);
  };
  auto saved = [&](int g, int i, int c) -> f32x4& { return slot(lds + g * GRP + 2 * BUF, i, c); };
  auto partial = [&](int g, int i, int c) -> f32x4& { return slot(lds + g * GRP, i, c); };
  // G = 2^lg (one share a group: the launch takes the tile only where G is WK)
  const int lg = MS > 1 ? k_shares_log2(nsc, N) : WK == 8 ? 3 : 2;
  int sh = (kg << lg) / WK, kend = nsc * (sh + 1) >> lg;  // the share that holds the next block, and its end
  while (kend <= k0 && kend < k1) kend = nsc * (++sh + 1) >> lg;  // (shares of short rows can be empty)
  bool kept = false;  // a share's sums are in `saved`
  auto chunk = [&](int i, int c) { return f32x4{acc[i][4 * c], acc[i][4 * c + 1], acc[i][4 * c + 2], acc[i][4 * c + 3]}; };
  auto add_saved = [&] {  // acc = saved + acc, the reads all in flight together
    f32x4 o[MT][4];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c) o[i][c] = saved(0, i, c);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][r] = o[i][r >> 2][r & 3] + acc[i][r];
  };

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
      if constexpr (MS > 1) {
        if (kb + 1 == kend && kend < k1) {  // the share ends here, and the group has another one
          if (WK == 1 && kept) add_saved();  // (a group that holds all of K adds its shares as it goes)
#pragma unroll
          for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
              saved(kg, i, c) = chunk(i, c);
#pragma unroll
              for (int r = 0; r < 4; ++r) acc[i][4 * c + r] = 0.f;
            }
          kept = true;
          do kend = nsc * (++sh + 1) >> lg;
          while (kend <= kb + 1);
        }
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
  if constexpr (WK > 1) {
    // The groups' sums, added in share order: group c adds and writes
    // chunk c, so a lane reads G 16-byte words (swiglu: twice that) in a row
    // and not, as one group adding them all would, 16 (WK - 1) registers.
    static_assert(WK >= NC && MS <= 2, "a group per chunk");
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c) partial(kg, i, c) = chunk(i, c);  // (over the buffers: all reads are done)
    lds_barrier();
    f32x4 g[MT], u[MT];
    if (kg < NC) {
      auto total = [&](int i, int c) {
        f32x4 p[WK], t;
#pragma unroll
        for (int k = 0; k < WK; ++k) p[k] = partial(k, i, c);
        if (kept) {  // two shares a group (of 32 blocks and more: none is empty)
          f32x4 v[WK];
#pragma unroll
          for (int k = 0; k < WK; ++k) v[k] = saved(k, i, c);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            t[r] = v[0][r] + p[0][r];
#pragma unroll
            for (int k = 1; k < WK; ++k) t[r] = (t[r] + v[k][r]) + p[k][r];
          }
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            t[r] = p[0][r];
#pragma unroll
            for (int k = 1; k < WK; ++k) t[r] = t[r] + p[k][r];
          }
        }
        return t;
      };
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        g[i] = total(i, kg);
        if constexpr (SW) u[i] = total(i, kg + 2);
      }
    }
    if (quant) lds_barrier();  // every read of the partial sums is done
    if (kg < NC) {
#pragma unroll
      for (int i = 0; i < MT; ++i) emit(i, kg, g[i], u[i]);
    }
  } else {
    if (kept) add_saved();
    if (quant) lds_barrier();  // every read of the saved sums is done
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

template <int MT, int WN, int WK, int MS>
void by_mode(int mode, const T32Args& a, int grid, hipStream_t st) {  // (a by reference: the grid's computation sets it)
  const dim3 blk(64 * WN * WK);
  if (a.dump)
    hipLaunchKernelGGL((gemm_t32_kernel<MT, WN, WK, 1, BTF_GEMV_STORE, true>), dim3(grid), blk, 0, st, a);
  else if (mode == BTF_GEMV_STORE)
    hipLaunchKernelGGL((gemm_t32_kernel<MT, WN, WK, MS, BTF_GEMV_STORE, false>), dim3(grid), blk, 0, st, a);
  else if (mode == BTF_GEMV_ADD)
    hipLaunchKernelGGL((gemm_t32_kernel<MT, WN, WK, MS, BTF_GEMV_ADD, false>), dim3(grid), blk, 0, st, a);
  else
    hipLaunchKernelGGL((gemm_t32_kernel<MT, WN, WK, MS, BTF_GEMV_SWIGLU, false>), dim3(grid), blk, 0, st, a);
}

// Output rows of a wave.
constexpr int t32_rows(int mode) { return mode == BTF_GEMV_SWIGLU ? 16 : 32; }

struct T32Tile {
  int mt, wn, wk;  // mt 0: no outputs
};

// Tile by the number of 32 x 32 output tiles per CU (a tile is a wave's work; a
// CU holds 16 waves at 4 per SIMD). Many: 64 activation rows per wave halve
// the decode per output, K unsplit. Fewer: 32 rows, and K split over the
// groups of a workgroup so that every SIMD has waves to overlap. The bits of y
// are the same in all of them. Measured on 256 CUs (us; tiles; the chosen one
// first):
//  - from 32 per CU: gate+up 5120 -> 2 x 17408, 512 rows (17408) 2,4,1 248,
//    1,4,1 273, 1,2,4 316; 256 rows (8704) 2,4,1 140, 1,4,1 146; 5120 -> 8192,
//    1024 rows (8192) 2,4,1 123, 1,4,1 138; below: gate+up, 224 rows (7616)
//    1,4,1 130, 2,4,1 139; 5120 -> 8192, 800 rows (6400) 1,4,1 116, 2,4,1 120;
//  - from 10 per CU K unsplit: 600 rows of 5120 -> 5120 (3040) 1,4,1 55.8, 1,2,4
//    60.0; 544 rows (2720) 54.0 / 57.9; 160 rows of 5120 -> 17408 (2720) 53.2 / 56.4;
//    3072 -> 5376, 512 rows (2688) 35.5 / 37.4; below: 5120 -> 5120, 512 rows (2560)
//    1,2,4 50.2, 1,4,1 52.9; gate+up, 64 rows (2176) 48.7 / 51.1; down 17408 ->
//    5120, 203 rows (1120) 94.7 / 118;
//  - from 4 per CU where a group would have one block at most: 256 -> 4096, 320
//    rows (1280) 1,4,1 5.3, 1,1,4 6.3, 1,2,4 7.5; 384 -> 4096, 512 rows (2048)
//    7.2 / 9.2 / 9.3; below: 512 -> 3 x 4096, 64 rows (768) 1,1,4 4.8, 1,2,4 5.6,
//    1,4,1 6.4;
//  - up to one per CU a workgroup of one tile, on as many CUs as there are tiles:
//    32 rows of 5120 -> 5120 (160) 1,1,8 9.5, 1,2,8 12.9; 4096 -> 8192 (256) 8.8 /
//    11.6; down (160) 28.4 / 35.6; 2048 -> 8192 (256) 1,1,4 6.0, 1,2,4 7.4; 1024 ->
//    1024 (32) 4.2 / 5.3;
//  - up to two per CU eight groups where K has eight shares: 5120 -> 3 x 5120, 32
//    rows (480) 1,2,8 14.7, 1,2,4 15.6; 8192 -> 8192, 64 rows (512) 20.5 / 21.2; 4096
//    -> 2 x 4096, 40 rows (512) 11.9 / 12.8; past that 5120 -> 5120, 128 rows (640)
//    1,2,4 21.7, 1,2,8 24.9; 17408 -> 5120, 128 rows (640) 59.6 / 71.6.
T32Tile t32_tile(const int (&N)[3], int K, int nb, int mode, bool q8, int64_t cus) {
  int64_t n = 0;
  bool eight = true;  // every matrix has eight shares of K
  for (int i = 0; i < 3; ++i) {
    n += (N[i] + t32_rows(mode) - 1) / t32_rows(mode);
    eight = eight && (N[i] == 0 || k_shares_log2(K / 128, N[i]) == 3);
  }
  const int64_t t32 = n * ((nb + 31) / 32);
  const bool wide = q8 && mode == BTF_GEMV_SWIGLU;  // (its Q8 blocks are two waves wide)
  if (t32 == 0) return {0, 0, 0};
  if (t32 >= 32 * cus && nb > 32) return {2, 4, 1};
  if (t32 > 10 * cus || (K <= 512 && t32 >= 4 * cus)) return {1, 4, 1};
  if (eight && t32 <= cus && !wide) return {1, 1, 8};
  if (eight && t32 <= 2 * cus) return {1, 2, 8};
  if (K < 4096 && (t32 <= cus || K <= 512) && !wide) return {1, 1, 4};
  return {1, 2, 4};
}

}  // namespace

int gemm_t32_tile(const int (&N)[3], int K, int nb, int mode, bool q8, int cus) {
  const T32Tile t = t32_tile(N, K, nb, mode, q8, cus);
  return 10000 * t.mt + 100 * t.wn + t.wk;
}

int gemm_t32(const GemvSeg* segs, int nseg, int K, int m0, int nb, const Q8& act, int mode, int32_t* dump,
             hipStream_t st, const DevState& ds, const Q8* qout) {
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
  const int N[3] = {nuse > 0 ? segs[0].N : 0, nuse > 1 ? segs[1].N : 0, nuse > 2 ? segs[2].N : 0};
  const T32Tile t = t32_tile(N, K, nb, mode, qout != nullptr, ds.cu_count);
  if (t.mt == 0) return BTF_OK;
  const int grid = tiles(t.wn * t32_rows(mode), 32 * t.mt);
  bool four = true;  // every matrix has four shares of K: one for each of four groups
  for (int i = 0; i < nuse; ++i) four = four && (N[i] == 0 || k_shares_log2(K / 128, N[i]) == 2);
  if (t.mt == 2)
    by_mode<2, 4, 1, 8>(mode, a, grid, st);
  else if (t.wn == 4)
    by_mode<1, 4, 1, 8>(mode, a, grid, st);
  else if (t.wn == 2 && t.wk == 8)
    by_mode<1, 2, 8, 1>(mode, a, grid, st);
  else if (t.wn == 2 && four)  // (1152 -> 16000, 32 rows: 5.98 us, 6.25 with the instance that sets sums aside)
    by_mode<1, 2, 4, 1>(mode, a, grid, st);
  else if (t.wn == 2)
    by_mode<1, 2, 4, 2>(mode, a, grid, st);
  else if (t.wk == 8)
    by_mode<1, 1, 8, 1>(mode, a, grid, st);
  else
    by_mode<1, 1, 4, 1>(mode, a, grid, st);
  return launch_status("gemm_t32_kernel");
}

}  // namespace btfhip
