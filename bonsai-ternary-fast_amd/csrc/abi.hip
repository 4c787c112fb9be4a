// abi.hip -- the extern "C" boundary (include/btf/hip_abi.h): host-side
// argument checks, per-device state, path dispatch and a small runtime shim.
// Argument checks mirror the reference launchers (src/cuda/kernels.cu:737-822)
// and run before any HIP call, so a CPU-only process can exercise them.
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>

#include "../../include/btf/hip_abi.h"
#include "common.h"

namespace btfhip {

namespace {
thread_local std::string g_err;
constexpr int kMaxDevices = 64;
DevState g_dev[kMaxDevices];
std::mutex g_init_mu;
// Batches of M >= this many rows use the int8-MFMA kernel.
constexpr int kDefaultMfmaMinM = 3;
int g_mfma_min_m = kDefaultMfmaMinM;

bool aligned(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }
}  // namespace

void set_error(const std::string& msg) { g_err = msg; }

int fail(int code, const std::string& msg) {
  g_err = msg;
  return code;
}

int launch_status(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(BTF_ERR_LAUNCH, std::string(what) + ": " + hipGetErrorString(e));
  return BTF_OK;
}

DevState* dev_state(int device) {
  if (device < 0 || device >= kMaxDevices) return nullptr;
  return &g_dev[device];
}

const DevState* current_state() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    set_error("no current HIP device");
    return nullptr;
  }
  if (!g_dev[dev].init) {
    set_error("btf_hip_kernels_init was not called for device " + std::to_string(dev));
    return nullptr;
  }
  return &g_dev[dev];
}

}  // namespace btfhip

using namespace btfhip;

namespace {

int hip_call(hipError_t e, const char* what) {
  if (e != hipSuccess) return fail(BTF_ERR_LAUNCH, std::string(what) + ": " + hipGetErrorString(e));
  return BTF_OK;
}

int check_q8(const btf_q8act* a, const char* who) {
  if (!a || !a->q || !a->d || !a->s) return fail(BTF_ERR_ARGS, std::string(who) + ": null activation pointer");
  if (!aligned(a->q, 16) || !aligned(a->d, 8) || !aligned(a->s, 8))
    return fail(BTF_ERR_ARGS, std::string(who) + ": q must be 16-byte and d/s 8-byte aligned");
  return BTF_OK;
}

// Shared checks of launch_gemv / gemv_i32_dump (src/cuda/kernels.cu:777-782).
int check_gemv(const btf_gemv_seg* segs, int nseg, int K, int M, const btf_q8act* a, int mode, bool need_y) {
  if (!segs) return fail(BTF_ERR_ARGS, "gemv: null segments");
  if (nseg < 1 || nseg > 3) return fail(BTF_ERR_ARGS, "gemv: 1..3 segments");
  if (mode != BTF_GEMV_STORE && mode != BTF_GEMV_ADD && mode != BTF_GEMV_SWIGLU)
    return fail(BTF_ERR_ARGS, "gemv: unknown mode");
  if (mode == BTF_GEMV_SWIGLU && (nseg != 2 || segs[0].N != segs[1].N))
    return fail(BTF_ERR_ARGS, "gemv: swiglu needs gate+up");
  if (K <= 0 || K % 128) return fail(BTF_ERR_ARGS, "gemv: K must be a multiple of 128");
  const int nuse = mode == BTF_GEMV_SWIGLU ? 2 : nseg;
  for (int i = 0; i < nuse; ++i) {
    const btf_gemv_seg& s = segs[i];
    if (s.N < 0) return fail(BTF_ERR_ARGS, "gemv: negative N");
    if (s.N == 0) continue;
    if (!s.codes || !s.scales) return fail(BTF_ERR_ARGS, "gemv: null weight pointer");
    if (!aligned(s.codes, 16) || !aligned(s.scales, 2))
      return fail(BTF_ERR_ARGS, "gemv: codes must be 16-byte aligned");
    const bool has_y = mode != BTF_GEMV_SWIGLU || i == 0;
    if (need_y && has_y) {
      if (!s.y) return fail(BTF_ERR_ARGS, "gemv: null output");
      if (M > 1 && s.ldy < s.N) return fail(BTF_ERR_ARGS, "gemv: ldy < N");
    }
  }
  return check_q8(a, "gemv");
}

int run_gemv(const btf_gemv_seg* segs, int nseg, int K, int M, const btf_q8act* act, int mode, int32_t* dump,
             hipStream_t st) {
  const DevState* ds = current_state();
  if (!ds) return BTF_ERR_NOT_INIT;
  GemvSeg sg[3];
  for (int i = 0; i < nseg; ++i) sg[i] = {segs[i].codes, segs[i].scales, segs[i].N, segs[i].y, segs[i].ldy};
  const Q8 a{act->q, act->d, act->s};
  // int8-MFMA path for larger batches and for rows wider than the dot4
  // workgroup covers (K > 32768).
  if (M >= g_mfma_min_m || K > 32768) return gemm_mfma(sg, nseg, K, 0, M, a, mode, dump, st, *ds);
  // v_dot4 path: up to 4 activation rows per pass; 2 past K = 16384 (down of two rows 21.2 us
  // in two passes, 16.0 in one), 1 past K = 20480.
  const int per = K > 20480 ? 1 : K > 16384 ? 2 : 4;
  for (int m0 = 0; m0 < M; m0 += per) {
    const int nb = M - m0 < per ? M - m0 : per;
    const int rc = gemv_dot4(sg, nseg, K, m0, nb, a, mode, dump, st, *ds);
    if (rc != BTF_OK) return rc;
  }
  return BTF_OK;
}

}  // namespace

extern "C" {

int btf_hip_kernels_init(int device) {
  DevState* s = dev_state(device);
  if (!s) return fail(BTF_ERR_DEVICE, "kernels_init: device id out of range");
  std::lock_guard<std::mutex> lk(g_init_mu);
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || device >= n)
    return fail(BTF_ERR_DEVICE, "kernels_init: no HIP device " + std::to_string(device));
  hipDeviceProp_t p;
  if (hipGetDeviceProperties(&p, device) != hipSuccess) return fail(BTF_ERR_DEVICE, "kernels_init: device query");
  s->cu_count = p.multiProcessorCount;
  s->lds_per_block = (int)p.sharedMemPerBlock;
  s->max_threads = p.maxThreadsPerBlock;
  if (!s->argmax_scratch) {  // the static scratch's address on this device (with the device current)
    int cur = -1;
    if (hipGetDevice(&cur) != hipSuccess) return fail(BTF_ERR_DEVICE, "kernels_init: hipGetDevice");
    if (cur != device && hipSetDevice(device) != hipSuccess) return fail(BTF_ERR_DEVICE, "kernels_init: hipSetDevice");
    const int rc = argmax_scratch_setup(*s);
    if (cur != device) (void)hipSetDevice(cur);
    if (rc != BTF_OK) return rc;
  }
  s->init = true;
  return BTF_OK;
}

int btf_hip_gemv_max_nb(int K) {
  if (K <= 0 || K % 128) return 0;
  return mfma_rows_per_pass();
}

int btf_hip_launch_repack(const uint8_t* src, int64_t nblocks, uint8_t* codes, uint16_t* scales,
                          btf_stream_t stream) {
  if (nblocks <= 0) return BTF_OK;
  if (!src || !codes || !scales) return fail(BTF_ERR_ARGS, "repack: null pointer");
  if (!aligned(src, 4) || !aligned(codes, 16) || !aligned(scales, 2))
    return fail(BTF_ERR_ARGS, "repack: src must be 4-byte and codes 16-byte aligned");
  const DevState* ds = current_state();
  if (!ds) return BTF_ERR_NOT_INIT;
  return repack(src, nblocks, codes, scales, static_cast<hipStream_t>(stream), *ds);
}

int btf_hip_launch_prep(const float* x, int ldx, int M, int n, const float* normw, float eps, const btf_hx* hx,
                        float* xn_out, int ldxn, const btf_q8act* a, btf_stream_t stream) {
  if (M <= 0) return BTF_OK;
  if (n <= 0 || n % 32) return fail(BTF_ERR_ARGS, "prep: width must be a multiple of 32");
  if (!x || ldx < n) return fail(BTF_ERR_ARGS, "prep: bad input (null x or ldx < n)");
  if (xn_out && ldxn < n) return fail(BTF_ERR_ARGS, "prep: ldxn < n");
  const int rc = check_q8(a, "prep");
  if (rc != BTF_OK) return rc;
  const int block = hx ? hx->block : 0;
  if (block < 0 || (block > 0 && (block & (block - 1))))
    return fail(BTF_ERR_ARGS, "prep: hadamard block must be 0 or a power of two");
  if (block > 0 && n % block) return fail(BTF_ERR_ARGS, "prep: hadamard block does not divide the width");
  if (block > 0 && hx->perm_rep > 1 && (int64_t)hx->perm_hd * hx->perm_nk * hx->perm_rep != n)
    return fail(BTF_ERR_ARGS, "prep: hadamard perm geometry");
  const DevState* ds = current_state();
  if (!ds) return BTF_ERR_NOT_INIT;
  return prep(x, ldx, M, n, normw, eps, block, hx ? hx->perm_hd : 0, hx ? hx->perm_nk : 0, hx ? hx->perm_rep : 0,
              hx ? hx->signs : nullptr, xn_out, ldxn, a->q, a->d, a->s, static_cast<hipStream_t>(stream), *ds);
}

int btf_hip_launch_gemv(const btf_gemv_seg* segs, int nseg, int K, int M, const btf_q8act* a, int mode,
                        btf_stream_t stream) {
  if (M <= 0) return BTF_OK;
  const int rc = check_gemv(segs, nseg, K, M, a, mode, true);
  if (rc != BTF_OK) return rc;
  return run_gemv(segs, nseg, K, M, a, mode, nullptr, static_cast<hipStream_t>(stream));
}

int btf_hip_launch_embed(const uint8_t* codes, const uint16_t* scales, const int* d_tok, int M, int E,
                         const btf_hx* inv, float* x, btf_stream_t stream) {
  if (M <= 0) return BTF_OK;
  if (!codes || !scales || !d_tok || !x) return fail(BTF_ERR_ARGS, "embed: null pointer");
  if (E <= 0 || E % 128) return fail(BTF_ERR_ARGS, "embed: width must be a multiple of 128");
  if (!aligned(codes, 4) || !aligned(scales, 2)) return fail(BTF_ERR_ARGS, "embed: codes must be 4-byte aligned");
  const int block = inv ? inv->block : 0;
  if (block < 0 || (block > 0 && (block & (block - 1))))
    return fail(BTF_ERR_ARGS, "embed: hadamard block must be 0 or a power of two");
  const DevState* ds = current_state();
  if (!ds) return BTF_ERR_NOT_INIT;
  return embed(codes, scales, d_tok, M, E, block, inv ? inv->signs : nullptr, x, static_cast<hipStream_t>(stream));
}

int64_t btf_hip_argmax_part_bytes(int V) { return argmax_part_bytes(V); }

int btf_hip_launch_argmax(const float* logits, int V, void* part, int* d_tok_out, btf_stream_t stream) {
  if (!logits || !part || !d_tok_out) return fail(BTF_ERR_ARGS, "argmax: null pointer");
  if (V <= 0) return fail(BTF_ERR_ARGS, "argmax: empty vocabulary");
  if (!aligned(part, 8)) return fail(BTF_ERR_ARGS, "argmax: part must be 8-byte aligned");
  const DevState* ds = current_state();
  if (!ds) return BTF_ERR_NOT_INIT;
  return argmax(logits, V, part, d_tok_out, static_cast<hipStream_t>(stream));
}

int btf_hip_launch_argmax_noalloc(const float* logits, int V, int* d_tok_out, btf_stream_t stream) {
  if (!logits || !d_tok_out) return fail(BTF_ERR_ARGS, "argmax_noalloc: null pointer");
  if (V <= 0) return fail(BTF_ERR_ARGS, "argmax_noalloc: empty vocabulary");
  const DevState* ds = current_state();
  if (!ds) return BTF_ERR_NOT_INIT;
  return argmax_noalloc(logits, V, d_tok_out, static_cast<hipStream_t>(stream), *ds);
}

int btf_hip_launch_pos_add(int* d_pos, int M, btf_stream_t stream) {
  if (!d_pos) return fail(BTF_ERR_ARGS, "pos_add: null pointer");
  const DevState* ds = current_state();
  if (!ds) return BTF_ERR_NOT_INIT;
  return pos_add(d_pos, M, static_cast<hipStream_t>(stream));
}

int btf_hip_launch_gemv_ex(const btf_gemv_seg* segs, int nseg, int K, int M, const btf_q8act* a, const float* x,
                           int ldx, int mode, const btf_q8act* out, btf_stream_t stream) {
  if (M <= 0) return BTF_OK;
  if ((a == nullptr) == (x == nullptr)) return fail(BTF_ERR_ARGS, "gemv_ex: give exactly one of a (Q8 rows) and x");
  if (x && (!aligned(x, 16) || ldx < K || ldx % 4))
    return fail(BTF_ERR_ARGS, "gemv_ex: x must be 16-byte aligned with ldx >= K and ldx % 4 == 0");
  if (K > 32768) return fail(BTF_ERR_ARGS, "gemv_ex: K > 32768");
  // the weight and output checks of launch_gemv (with x, the Q8 pointers are not read)
  const btf_q8act none{reinterpret_cast<int8_t*>(16), reinterpret_cast<float*>(16), reinterpret_cast<int32_t*>(16)};
  int rc = check_gemv(segs, nseg, K, M, a ? a : &none, mode, true);
  if (rc != BTF_OK) return rc;
  if (out) {
    if ((rc = check_q8(out, "gemv_ex")) != BTF_OK) return rc;
    if (mode != BTF_GEMV_SWIGLU && nseg != 1) return fail(BTF_ERR_ARGS, "gemv_ex: a Q8 output takes one segment");
    if (segs[0].N % 32) return fail(BTF_ERR_ARGS, "gemv_ex: a Q8 output needs N % 32 == 0");
  }
  const DevState* ds = current_state();
  if (!ds) return BTF_ERR_NOT_INIT;
  GemvSeg sg[3];
  for (int i = 0; i < nseg; ++i) sg[i] = {segs[i].codes, segs[i].scales, segs[i].N, segs[i].y, segs[i].ldy};
  const Q8 in = a ? Q8{a->q, a->d, a->s} : Q8{nullptr, nullptr, nullptr};
  const Q8 qo = out ? Q8{out->q, out->d, out->s} : Q8{nullptr, nullptr, nullptr};
  // Q8 rows in, Q8 rows out, a batch on the int8-MFMA path: one launch (32-row output tiles)
  if (a && out && M >= g_mfma_min_m && M <= 32)
    return gemm_mfma(sg, nseg, K, 0, M, in, mode, nullptr, static_cast<hipStream_t>(stream), *ds, &qo);
  for (int m = 0; m < M; ++m) {
    rc = gemv_dot4(sg, nseg, K, m, 1, in, mode, nullptr, static_cast<hipStream_t>(stream), *ds, x, ldx,
                   out ? &qo : nullptr);
    if (rc != BTF_OK) return rc;
  }
  return BTF_OK;
}

int btf_hip_launch_gemv_ptq1_0(const btf_gemv_seg* segs, int nseg, int K, int M, const btf_q8act* a, int mode,
                               btf_stream_t stream) {
  if (M <= 0) return BTF_OK;
  if (!segs) return fail(BTF_ERR_ARGS, "gemv_ptq1_0: null segments");
  if (K > 32768) return fail(BTF_ERR_ARGS, "gemv_ptq1_0: K > 32768");
  // the checks of launch_gemv, with the blocks' own scales (a placeholder passes the scale check)
  // (16-byte placeholders pass the T2 alignment checks; the blocks need 4 bytes)
  btf_gemv_seg sv[3];
  for (int i = 0; i < nseg && i < 3; ++i) {
    sv[i] = segs[i];
    if (segs[i].N == 0) continue;
    if (segs[i].scales) return fail(BTF_ERR_ARGS, "gemv_ptq1_0: scales must be NULL (they are inside the blocks)");
    if (!aligned(segs[i].codes, 4)) return fail(BTF_ERR_ARGS, "gemv_ptq1_0: blocks must be 4-byte aligned");
    sv[i].codes = segs[i].codes ? reinterpret_cast<const uint8_t*>(16) : nullptr;
    sv[i].scales = reinterpret_cast<const uint16_t*>(16);
  }
  int rc = check_gemv(sv, nseg, K, M, a, mode, true);
  if (rc != BTF_OK) return rc;
  const DevState* ds = current_state();
  if (!ds) return BTF_ERR_NOT_INIT;
  GemvSeg sg[3];
  for (int i = 0; i < nseg; ++i) sg[i] = {segs[i].codes, nullptr, segs[i].N, segs[i].y, segs[i].ldy};
  const Q8 q{a->q, a->d, a->s};
  for (int m0 = 0; m0 < M; m0 += 2) {
    rc = gemv_b3(sg, nseg, K, m0, M - m0 < 2 ? M - m0 : 2, q, mode, static_cast<hipStream_t>(stream), *ds);
    if (rc != BTF_OK) return rc;
  }
  return BTF_OK;
}

int btf_hip_gemv_i32_dump(const uint8_t* codes, int N, int K, int M, const btf_q8act* a, int32_t* I_out,
                          btf_stream_t stream) {
  if (M <= 0 || N <= 0) return BTF_OK;
  if (!I_out) return fail(BTF_ERR_ARGS, "gemv_i32_dump: null output");
  const btf_gemv_seg seg{codes, nullptr, N, nullptr, N};
  // scales are not read by the dump path; a non-null placeholder passes the check
  btf_gemv_seg s2 = seg;
  s2.scales = reinterpret_cast<const uint16_t*>(codes);
  const int rc = check_gemv(&s2, 1, K, M, a, BTF_GEMV_STORE, false);
  if (rc != BTF_OK) return rc;
  return run_gemv(&s2, 1, K, M, a, BTF_GEMV_STORE, I_out, static_cast<hipStream_t>(stream));
}

int btf_hip_gemv_set_policy(int mfma_min_m) {
  const int prev = g_mfma_min_m;
  g_mfma_min_m = mfma_min_m > 0 ? mfma_min_m : kDefaultMfmaMinM;
  return prev;
}

int btf_hip_gemm_tile(int cu_count, const int* N, int nseg, int K, int M, int mode, int q8_out) {
  if (!N || nseg < 1 || nseg > 3 || K <= 0 || K % 128 || M <= 16 || cu_count <= 0) return 0;
  int n[3] = {};
  for (int i = 0; i < (mode == BTF_GEMV_SWIGLU ? 1 : nseg); ++i) n[i] = N[i];
  return gemm_t32_tile(n, K, M, mode, q8_out != 0, cu_count);
}

int btf_hip_stream_read(const void* src, uint64_t bytes, uint32_t never, uint32_t* sink, btf_stream_t stream) {
  if (bytes == 0) return BTF_OK;
  if (!src || !sink || !aligned(src, 16) || bytes % 16)
    return fail(BTF_ERR_ARGS, "stream_read: src 16-byte aligned, bytes a multiple of 16, non-null sink");
  const DevState* ds = current_state();
  if (!ds) return BTF_ERR_NOT_INIT;
  return stream_read(src, bytes, never, sink, static_cast<hipStream_t>(stream), *ds);
}

int btf_hip_gen_ptq1_0(uint64_t seed, uint64_t mat, int64_t first_block, int64_t nblocks, uint8_t* dst,
                       btf_stream_t stream) {
  if (nblocks <= 0) return BTF_OK;
  if (!dst || !aligned(dst, 4)) return fail(BTF_ERR_ARGS, "gen_ptq1_0: dst must be 4-byte aligned");
  if (first_block < 0) return fail(BTF_ERR_ARGS, "gen_ptq1_0: negative first block");
  const DevState* ds = current_state();
  if (!ds) return BTF_ERR_NOT_INIT;
  return gen_ptq1_0(seed, mat, first_block, nblocks, dst, static_cast<hipStream_t>(stream), *ds);
}

int btf_hip_step_create(const btf_step_vec* vecs, int nvec, const btf_step_gemv* ops, int nops, btf_step_t* out) {
  if (!vecs || !ops || !out || nvec <= 0 || nops <= 0) return fail(BTF_ERR_ARGS, "step: empty program");
  if (const int rc = step_validate(vecs, nvec, ops, nops)) return rc;
  const DevState* ds = current_state();
  if (!ds) return BTF_ERR_NOT_INIT;
  StepProgram* P = nullptr;
  const int rc = step_create(vecs, nvec, ops, nops, &P, *ds);
  if (rc == BTF_OK) *out = P;
  return rc;
}

int btf_hip_step_create_ops(const btf_step_vec* vecs, int nvec, const btf_step_op* ops, int nops, btf_step_t* out) {
  if (!vecs || !ops || !out || nvec <= 0 || nops <= 0) return fail(BTF_ERR_ARGS, "step: empty program");
  if (const int rc = step_validate_ops(vecs, nvec, ops, nops)) return rc;
  const DevState* ds = current_state();
  if (!ds) return BTF_ERR_NOT_INIT;
  StepProgram* P = nullptr;
  const int rc = step_create_ops(vecs, nvec, ops, nops, &P, *ds);
  if (rc == BTF_OK) *out = P;
  return rc;
}

int btf_hip_step_audit(const btf_step_vec* vecs, int nvec, const btf_step_op* ops, int nops, int G,
                       btf_step_audit* out) {
  if (!vecs || !ops || !out || nvec <= 0 || nops <= 0) return fail(BTF_ERR_ARGS, "step: empty program");
  return step_audit(vecs, nvec, ops, nops, G, out);
}

int btf_hip_step_launch(btf_step_t prog, btf_stream_t stream) {
  if (!prog) return fail(BTF_ERR_ARGS, "step: null program");
  return step_launch(static_cast<StepProgram*>(prog), static_cast<hipStream_t>(stream));
}

int btf_hip_step_error(btf_step_t prog, int* error) {
  if (!prog || !error) return fail(BTF_ERR_ARGS, "step: null argument");
  return step_error(static_cast<StepProgram*>(prog), error);
}

int btf_hip_step_set_spin_limit(btf_step_t prog, uint32_t polls) {
  if (!prog) return fail(BTF_ERR_ARGS, "step: null program");
  return step_set_spin_limit(static_cast<StepProgram*>(prog), polls);
}

int btf_hip_step_guards(btf_step_t prog, int* guards) {
  if (!prog || !guards) return fail(BTF_ERR_ARGS, "step: null argument");
  return step_guards(static_cast<StepProgram*>(prog), guards);
}

int btf_hip_step_destroy(btf_step_t prog) {
  step_destroy(static_cast<StepProgram*>(prog));
  return BTF_OK;
}

const char* btf_hip_last_error(void) { return g_err.c_str(); }

int btf_hip_device_info(int device, btf_device_info* out) {
  if (!out) return fail(BTF_ERR_ARGS, "device_info: null output");
  hipDeviceProp_t p;
  if (hipGetDeviceProperties(&p, device) != hipSuccess) return fail(BTF_ERR_DEVICE, "device_info: device query");
  std::memset(out, 0, sizeof *out);
  out->cu_count = p.multiProcessorCount;
  out->lds_bytes_per_block = (int)p.sharedMemPerBlock;
  out->max_clock_khz = p.clockRate;
  out->mem_clock_khz = p.memoryClockRate;
  out->mem_bus_width_bits = p.memoryBusWidth;
  out->l2_bytes = p.l2CacheSize;
  out->wavefront_size = p.warpSize;
  out->arch_major = p.major;
  out->arch_minor = p.minor;
  out->total_mem_bytes = (int64_t)p.totalGlobalMem;
  std::snprintf(out->name, sizeof out->name, "%s", p.name);
  std::snprintf(out->gcn_arch, sizeof out->gcn_arch, "%s", p.gcnArchName);
  return BTF_OK;
}

// ---- runtime shim ----
int btf_hip_device_count(int* n) { return hip_call(hipGetDeviceCount(n), "hipGetDeviceCount"); }
int btf_hip_set_device(int device) { return hip_call(hipSetDevice(device), "hipSetDevice"); }
int btf_hip_malloc(void** p, size_t bytes) { return hip_call(hipMalloc(p, bytes), "hipMalloc"); }
int btf_hip_free(void* p) { return hip_call(hipFree(p), "hipFree"); }
int btf_hip_host_alloc_mapped(void** host, void** dev, size_t bytes) {
  int rc = hip_call(hipHostMalloc(host, bytes, hipHostMallocMapped), "hipHostMalloc");
  if (rc != BTF_OK) return rc;
  return hip_call(hipHostGetDevicePointer(dev, *host, 0), "hipHostGetDevicePointer");
}
int btf_hip_host_free(void* host) { return hip_call(hipHostFree(host), "hipHostFree"); }
int btf_hip_memcpy_h2d(void* dst, const void* src, size_t bytes) {
  return hip_call(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice), "hipMemcpy H2D");
}
int btf_hip_memcpy_d2h(void* dst, const void* src, size_t bytes) {
  return hip_call(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost), "hipMemcpy D2H");
}
int btf_hip_memset(void* dst, int value, size_t bytes) { return hip_call(hipMemset(dst, value, bytes), "hipMemset"); }
int btf_hip_device_synchronize(void) { return hip_call(hipDeviceSynchronize(), "hipDeviceSynchronize"); }
int btf_hip_stream_create(btf_stream_t* s) {
  hipStream_t h = nullptr;
  const int rc = hip_call(hipStreamCreateWithFlags(&h, hipStreamNonBlocking), "hipStreamCreate");
  *s = h;
  return rc;
}
int btf_hip_stream_destroy(btf_stream_t s) {
  return hip_call(hipStreamDestroy(static_cast<hipStream_t>(s)), "hipStreamDestroy");
}
int btf_hip_stream_synchronize(btf_stream_t s) {
  return hip_call(hipStreamSynchronize(static_cast<hipStream_t>(s)), "hipStreamSynchronize");
}
int btf_hip_event_create(btf_event_t* e) {
  hipEvent_t h = nullptr;
  const int rc = hip_call(hipEventCreate(&h), "hipEventCreate");
  *e = h;
  return rc;
}
int btf_hip_event_destroy(btf_event_t e) { return hip_call(hipEventDestroy(static_cast<hipEvent_t>(e)), "hipEventDestroy"); }
int btf_hip_event_record(btf_event_t e, btf_stream_t s) {
  return hip_call(hipEventRecord(static_cast<hipEvent_t>(e), static_cast<hipStream_t>(s)), "hipEventRecord");
}
int btf_hip_event_elapsed_ms(float* ms, btf_event_t a, btf_event_t b) {
  return hip_call(hipEventElapsedTime(ms, static_cast<hipEvent_t>(a), static_cast<hipEvent_t>(b)),
                  "hipEventElapsedTime");
}
int btf_hip_graph_begin(btf_stream_t s) {
  return hip_call(hipStreamBeginCapture(static_cast<hipStream_t>(s), hipStreamCaptureModeThreadLocal),
                  "hipStreamBeginCapture");
}
int btf_hip_graph_end(btf_stream_t s, btf_graph_exec_t* out) {
  hipGraph_t g = nullptr;
  int rc = hip_call(hipStreamEndCapture(static_cast<hipStream_t>(s), &g), "hipStreamEndCapture");
  if (rc != BTF_OK) return rc;
  hipGraphExec_t ex = nullptr;
  rc = hip_call(hipGraphInstantiate(&ex, g, nullptr, nullptr, 0), "hipGraphInstantiate");
  (void)hipGraphDestroy(g);
  *out = ex;
  return rc;
}
int btf_hip_graph_launch(btf_graph_exec_t g, btf_stream_t s) {
  return hip_call(hipGraphLaunch(static_cast<hipGraphExec_t>(g), static_cast<hipStream_t>(s)), "hipGraphLaunch");
}
int btf_hip_graph_destroy(btf_graph_exec_t g) {
  return hip_call(hipGraphExecDestroy(static_cast<hipGraphExec_t>(g)), "hipGraphExecDestroy");
}

}  // extern "C"
