// Entry points of the key/value-gradient step of one chunk attention backward for gfx950, against an external
// (ring-combined) base-2 LSE and delta = rowsum(O*dO): argument checks, the head split and its reduction kernel. The
// kernels are attn_bwd_dkdv_d64.hip, attn_bwd_dkdv_d128.hip and attn_bwd_dkdv_d192.hip.
//
// With grouped-query attention the heads of a group may be cut into `split` parts handled by
// different workgroups (more parallelism when there are few key tiles); the parts leave fp32
// partial results in a caller-provided workspace and a second kernel adds them in a fixed
// order, so the result does not depend on scheduling.
#include <mutex>

#include "attn_bwd_common.h"

namespace pith {
namespace {

constexpr int kBN = kDkdvBlockN;  // key rows per workgroup

// out[b, s, h, :] (+)= sum over parts of ws[part][b][s][h][:], parts added in index order; dK
// (blockIdx.y = 0) and dV (blockIdx.y = 1) in one launch.
struct ReduceParams {
  const float* ws[2];
  void* out[2];
  int64_t part_stride[2], row_elems[2], out_bs[2], n4[2];
  int64_t out_row_elems[2];  // elements between consecutive rows of `out` (>= row_elems: a head range of a wider tensor)
  int64_t rows_per_batch;
  int parts, accumulate;
};

template <typename OutT>
__global__ __launch_bounds__(256) void reduce_parts_kernel(ReduceParams r) {
  const int t = blockIdx.y;
  const float* __restrict__ ws = r.ws[t];
  OutT* out = reinterpret_cast<OutT*>(r.out[t]);
  const int64_t part_stride = r.part_stride[t], n4 = r.n4[t];
  const int64_t per_batch = r.rows_per_batch * r.row_elems[t];
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t e = i * 4;
    f32x4 s = *reinterpret_cast<const f32x4*>(ws + e);
    for (int pidx = 1; pidx < r.parts; ++pidx) s += *reinterpret_cast<const f32x4*>(ws + pidx * part_stride + e);
    const int64_t bb = e / per_batch;
    const int64_t in_batch = e - bb * per_batch;
    const int64_t row = in_batch / r.row_elems[t];
    OutT* dst = out + bb * r.out_bs[t] + row * r.out_row_elems[t] + (in_batch - row * r.row_elems[t]);
    store4<OutT>(dst, s[0], s[1], s[2], s[3], r.accumulate != 0);
  }
}

int pick_split(const pith_attn_bwd_args* a) {
  const int64_t group = a->Hq / a->Hkv;
  const int64_t base = ((a->Skv + kBN - 1) / kBN) * a->Hkv * a->B;
  int split = 1;
  // Workgroups wanted. Without a causal mask all of them carry the same work, so one full round is ideal; under the mask
  // two rounds (heaviest first) balance better. At 64 features two workgroups share a compute unit and twice as many are
  // wanted (8192 rows x 32 heads causal: 757 us with 512 workgroups, 560 us with 1024; without a mask 512 and 1024 are
  // within 2 %).
  const int64_t want = (a->causal ? 2 : 1) * (a->Dqk == 64 ? 2 : 1) * (int64_t)compute_units_or_default();
  while (split < group && base * split < want && group % (split * 2) == 0) split *= 2;
  return split;
}

// Workspace layout: [head-split partial dK | partial dV] (split > 1), then the per-head gradients of a
// shared k_pe [Hkv][B][Skv][64] (keys in two parts).
int64_t split_bytes_for(const pith_attn_bwd_args* a, int split) {
  if (split <= 1) return 0;
  return (int64_t)split * a->B * a->Skv * a->Hkv * (a->Dqk + a->Dv) * (int64_t)sizeof(float);
}
int64_t dkpe_bytes_for(const pith_attn_bwd_args* a) {
  return a->k_pe ? a->Hkv * a->B * a->Skv * 64 * (int64_t)sizeof(float) : 0;
}
int64_t workspace_bytes_for(const pith_attn_bwd_args* a, int split) { return split_bytes_for(a, split) + dkpe_bytes_for(a); }

constexpr int64_t kWalkDescBytes = 192ll << 20;

// with_dq: dQ of the pair in the same grid (p prepared for it)
template <int DQK, int DV>
void launch_dkdv(BwdParams p, const pith_attn_bwd_args* a, bool with_dq, hipStream_t st) {
  p.tiles = (int)((a->Skv + kBN - 1) / kBN);
  p.accumulate = a->accumulate_dkv;
  p.main_blocks = (int)(p.tiles * a->Hkv * a->B * p.split);
  p.zero_tail = a->accumulate_dkv ? 0 : (int)a->dkv_zero_tail;  // rows that are added to keep what they hold
  const unsigned grid = (unsigned)(p.main_blocks + (p.zero_tail + kZeroTailRows - 1) / kZeroTailRows);
  const bool f32 = a->dkv_dtype == PITH_F32;
  if (with_dq) {
    launch_bwd_pair(p, DQK, a->causal != 0, f32, a->dq_dtype == PITH_F32, grid, st);
  } else if constexpr (DQK == 128 && DV == 128) {
    // descending walk under the mask when Q and dO together exceed what the last-level cache (256 MB) keeps
    p.walk_desc = a->causal != 0 && (int64_t)a->B * a->Sq * a->Hq * (DQK + DV) * 2 > kWalkDescBytes;
    launch_dkdv_d128(p, a->causal != 0, f32, grid, st);
  } else if constexpr (DQK == 192 && DV == 128) {
    launch_dkdv_d192(p, a->causal != 0, f32, grid, st);
  } else {
    launch_dkdv_d64(p, a->causal != 0, f32, grid, st);
  }
  if (p.k_pe) {  // dk_pe (+)= sum over heads, in head order
    ReduceParams r;
    r.row_elems[0] = r.out_row_elems[0] = 64;
    r.part_stride[0] = a->B * a->Skv * 64;
    r.n4[0] = r.part_stride[0] / 4;
    r.ws[0] = p.ws_dkpe;
    r.out[0] = a->dk_pe;
    r.out_bs[0] = a->dk_pe_bs;
    r.row_elems[1] = r.out_row_elems[1] = r.part_stride[1] = r.n4[1] = r.out_bs[1] = 0;
    r.ws[1] = nullptr;
    r.out[1] = nullptr;
    r.rows_per_batch = a->Skv;
    r.parts = (int)a->Hkv;
    r.accumulate = a->accumulate_dkv;
    const int64_t blocks = (r.n4[0] + 255) / 256;
    const dim3 rgrid((unsigned)(blocks < 8192 ? blocks : 8192), 1);
    if (f32) hipLaunchKernelGGL((reduce_parts_kernel<float>), rgrid, dim3(256), 0, st, r);
    else hipLaunchKernelGGL((reduce_parts_kernel<__bf16>), rgrid, dim3(256), 0, st, r);
  }
  if (p.split > 1) {
    ReduceParams r;
    int64_t max_n4 = 0;
    for (int which = 0; which < 2; ++which) {
      const int64_t d = which == 0 ? a->Dqk : a->Dv;
      r.row_elems[which] = a->Hkv * d;
      r.out_row_elems[which] = p.HkvT * d;
      r.part_stride[which] = a->B * a->Skv * r.row_elems[which];
      r.n4[which] = r.part_stride[which] / 4;
      r.ws[which] = which == 0 ? p.ws_dk : p.ws_dv;
      r.out[which] = which == 0 ? a->dk : a->dv;
      r.out_bs[which] = which == 0 ? a->dk_bs : a->dv_bs;
      if (r.n4[which] > max_n4) max_n4 = r.n4[which];
    }
    r.rows_per_batch = a->Skv;
    r.parts = p.split;
    r.accumulate = a->accumulate_dkv;
    const dim3 rgrid((unsigned)((max_n4 + 255) / 256 < 8192 ? (max_n4 + 255) / 256 : 8192), 2);
    if (f32) hipLaunchKernelGGL((reduce_parts_kernel<float>), rgrid, dim3(256), 0, st, r);
    else hipLaunchKernelGGL((reduce_parts_kernel<__bf16>), rgrid, dim3(256), 0, st, r);
  }
}

}  // namespace
}  // namespace pith

using namespace pith;

extern "C" int64_t pith_attn_bwd_dkdv_workspace_bytes(const pith_attn_bwd_args* a) {
  if (!a || a->Hkv <= 0 || a->Hq <= 0 || a->Hq % a->Hkv != 0 || a->B <= 0 || a->Skv <= 0) return 0;
  return workspace_bytes_for(a, pick_split(a));
}

namespace {

// Runs the kernels with the head-split partials in `workspace` (NULL: no head split).
int run_dkdv(const pith_attn_bwd_args* a, int split, void* workspace, hipStream_t st, const char* who, bool with_dq = false) {
  // the grid of this kernel runs over key tiles (validate_bwd bounded the query-side grid)
  if (((a->Skv + kBN - 1) / kBN) * a->Hkv * a->B * (int64_t)split > 0x7fffffffLL)
    return fail(PITH_ERR_UNSUPPORTED, "%s: Skv=%lld x Hkv=%lld x B=%lld exceeds the launch grid limit", who,
                (long long)a->Skv, (long long)a->Hkv, (long long)a->B);
  BwdParams p = make_bwd_params(a);
  if (with_dq)
    if (const int rc = prepare_dq(a, &p, who)) return rc;
  if (a->k_pe) {
    if (a->Hq != a->Hkv)
      return fail(PITH_ERR_UNSUPPORTED, "%s: keys in two parts need Hq == Hkv (got %lld, %lld)", who, (long long)a->Hq, (long long)a->Hkv);
    if (!a->dk_pe) return fail(PITH_ERR_NULL_POINTER, "%s: dk_pe is NULL", who);
    if (!aligned16(a->dk_pe) || a->dk_pe_bs % 8) return fail(PITH_ERR_MISALIGNED, "%s: dk_pe pointer / batch stride must keep 16-byte alignment", who);
    if (!workspace) return fail(PITH_ERR_BAD_SHAPE, "%s: keys in two parts need a workspace of %lld bytes", who, (long long)dkpe_bytes_for(a));
    p.ws_dkpe = reinterpret_cast<float*>(reinterpret_cast<char*>(workspace) + split_bytes_for(a, split));
  }
  begin_launch();
  if (split > 1 && workspace) {
    p.split = split;
    p.ws_dk = reinterpret_cast<float*>(workspace);
    p.ws_dv = p.ws_dk + (int64_t)split * a->B * a->Skv * a->Hkv * a->Dqk;
  }
  // dS hand-over to the dQ call: only when the buffer is usable (otherwise the call behaves as without it)
  if (ds_usable(a)) {
    if ((uintptr_t)a->ds % 256) return fail(PITH_ERR_MISALIGNED, "%s: ds must be 256-byte aligned", who);
    p.ds = reinterpret_cast<char*>(a->ds);
  }
  if (a->Dqk == 128) launch_dkdv<128, 128>(p, a, with_dq, st);
  else if (a->Dqk == 192) launch_dkdv<192, 128>(p, a, with_dq, st);
  else launch_dkdv<64, 64>(p, a, with_dq, st);
  return check_launch(who);
}

// Scratch of pith_attn_bwd_dkdv_static: device memory that belongs to the library's code object
// (one copy per GPU, held until the process ends). Host code never uses this name as an address;
// it asks the runtime for the array's device address once per device and passes that on.
constexpr int64_t kStaticScratchBytes = PITH_DKDV_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device; resolved at the first call on that device.
int static_scratch(void** out, const char* who) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(PITH_ERR_LAUNCH, "%s: hipGetDevice: %s", who, hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices) return fail(PITH_ERR_UNSUPPORTED, "%s: device index %d beyond %d", who, dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
      return fail(PITH_ERR_LAUNCH, "%s: hipGetSymbolAddress(scratch) on device %d: %s", who, dev, hipGetErrorString(e));
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return PITH_OK;
}

}  // namespace

namespace {

int bwd_dkdv(const pith_attn_bwd_args* a, pith_stream_t stream, const char* who, bool with_dq) {
  const int rc = validate_bwd(a, who, false, true);
  if (rc != PITH_OK) return rc;
  // Head groups are split only when the caller brought a workspace that is large enough.
  int split = pick_split(a);
  if (!(split > 1 && a->workspace && a->workspace_bytes >= workspace_bytes_for(a, split))) split = 1;
  if (a->workspace && !aligned16(a->workspace)) return fail(PITH_ERR_MISALIGNED, "%s: workspace must be 16-byte aligned", who);
  if (a->k_pe && (!a->workspace || a->workspace_bytes < workspace_bytes_for(a, split)))
    return fail(PITH_ERR_BAD_SHAPE, "%s: keys in two parts need a workspace of %lld bytes, %lld given", who,
                (long long)workspace_bytes_for(a, split), (long long)(a->workspace ? a->workspace_bytes : 0));
  return run_dkdv(a, split, a->workspace, (hipStream_t)stream, who, with_dq);
}

// Whether dK/dV and dQ go out as one grid (no dS handed over). At 128 and 192 features the dQ workgroups are then the
// split-key ones (the two kernels must agree on the workgroup size), which is what grids of up to one workgroup per compute
// unit want anyway; larger ones fill the device with either kernel and gain nothing (1 x 4096 x 16 heads of 192 features,
// 512 + 512 workgroups: 293 us apart, 298 us together). At 64 features one kernel costs dQ its third workgroup per compute
// unit (186 instead of 150 registers), which only grids of a few rounds do not miss (1 x 4096 x 16 heads causal 184 -> 130 us,
// 1 x 4096 x 32 262 -> 259 us, 4 x 4096 x 16 474 -> 483 us).
bool one_grid(const pith_attn_bwd_args* a) {
  if (ds_usable(a) || (a->dkv_dtype == PITH_F32 && a->dq_dtype != PITH_F32)) return false;
  const int64_t q_wgs = ((a->Sq + 127) / 128) * a->Hq * a->B;
  return q_wgs <= (a->Dqk == 64 ? 4 : 1) * (int64_t)compute_units_or_default();
}

}  // namespace

extern "C" int pith_attn_bwd_dkdv(const pith_attn_bwd_args* a, pith_stream_t stream) {
  return bwd_dkdv(a, stream, "pith_attn_bwd_dkdv", false);
}

extern "C" int pith_attn_bwd(const pith_attn_bwd_args* a, pith_stream_t stream) {
  if (const int rc = validate_bwd(a, "pith_attn_bwd", true, true)) return rc;
  if (one_grid(a)) return bwd_dkdv(a, stream, "pith_attn_bwd", true);
  if (const int rc = pith_attn_bwd_dkdv(a, stream)) return rc;
  return pith_attn_bwd_dq(a, stream);
}

extern "C" int pith_attn_bwd_dkdv_static(const pith_attn_bwd_args* a, pith_stream_t stream) {
  const char* who = "pith_attn_bwd_dkdv_static";
  const int rc = validate_bwd(a, who, false, true);
  if (rc != PITH_OK) return rc;
  const int split = pick_split(a);
  const int64_t need = workspace_bytes_for(a, split);
  if (need > kStaticScratchBytes)
    return fail(PITH_ERR_UNSUPPORTED,
                "%s: the head-split partial sums of this shape need %lld bytes, the built-in scratch holds %lld "
                "(use pith_attn_bwd_dkdv with a caller-provided workspace)",
                who, (long long)need, (long long)kStaticScratchBytes);
  void* ws = nullptr;
  if (need > 0) {
    const int src = static_scratch(&ws, who);
    if (src != PITH_OK) return src;
  }
  return run_dkdv(a, split, ws, (hipStream_t)stream, who);
}
