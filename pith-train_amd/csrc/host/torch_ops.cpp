// The operators' host path in native code: torch.library ops with their autograd formulas, and the fast form of
// the *_into calls, both straight on top of the C ABI (include/pith_hip.h).
//
// What bounds a small call is the host, not the GPU: the kernels of a 256-token layer run for 50 us, while checking
// tensors, filling argument structs and dispatching through Python took 400 us a forward + backward. Everything here
// therefore works on at::Tensor directly, allocates from torch's caching allocator and enqueues on the current stream.
//
// Two layers share each operator. The native one serves the calls of ordinary layout (GPU tensors, the expected dtypes,
// contiguous per batch element). Whenever a condition fails, or the library rejects the arguments, it has launched nothing yet
// and hands over to the operator's Python body, which accepts every layout (copying where needed) and words the errors. A
// launch that fails is raised as it is (see accepted()).
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>
#include <torch/library.h>

#include <array>
#include <array>
#include <atomic>
#include <cstdlib>

#include "pith_hip.h"
#include "../handover_rows.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ---------------------------------------------------------------------------------------------
// Python bodies of the ops, registered once at import.
py::object& bodies() {
  static py::object* d = new py::object(py::dict());  // never destroyed: the interpreter may be gone by then
  return *d;
}

template <typename R, typename... Args>
R python_body(const char* name, const Args&... args) {
  py::gil_scoped_acquire gil;
  return bodies()[name](args...).template cast<R>();
}

// Whether the library took a call. One that it rejected has launched nothing, so the Python body may run it again. After a
// failed launch that is not so: kernels of the call may be out, and accumulating ones must not run twice. Raises PithError.
bool accepted(int rc) {
  if (rc == PITH_ERR_LAUNCH) python_body<bool>("check", rc);
  return rc == PITH_OK;
}

// ---------------------------------------------------------------------------------------------
// Layout checks, mirroring pithtrain_amd/_C.py. False: not a layout the native path takes.

bool is_gpu_bf16(const Tensor& t, int64_t dim) { return t.is_cuda() && t.scalar_type() == at::kBFloat16 && t.dim() == dim; }
bool is_gpu_f32(const Tensor& t, int64_t dim) { return t.is_cuda() && t.scalar_type() == at::kFloat && t.dim() == dim; }
bool has_shape(const Tensor& t, at::IntArrayRef shape) { return t.sizes() == shape; }

// [B, S, H, D], contiguous within a batch element (a slice along S of a contiguous tensor qualifies)
bool bshd(const Tensor& t, int64_t* batch_stride) {
  const auto n = t.sizes();
  const auto st = t.strides();
  if (!((n[3] == 1 || st[3] == 1) && (n[2] == 1 || st[2] == n[3]) && (n[1] == 1 || st[1] == n[2] * n[3]))) return false;
  *batch_stride = n[0] > 1 ? st[0] : n[1] * n[2] * n[3];
  return true;
}

// The same for what may be a range of consecutive heads of a wider tensor; heads per row of that tensor come back too.
bool bshd_heads(const Tensor& t, int64_t* batch_stride, int64_t* row_heads) {
  const auto n = t.sizes();
  const auto st = t.strides();
  const int64_t rh = n[1] == 1 ? n[2] : (n[3] > 0 ? st[1] / n[3] : 0);
  if (!((n[3] == 1 || st[3] == 1) && (n[2] == 1 || st[2] == n[3]) && (n[1] == 1 || (st[1] % n[3] == 0 && rh >= n[2])))) return false;
  *batch_stride = n[0] > 1 ? st[0] : n[1] * rh * n[3];
  *row_heads = rh;
  return true;
}

// [B, H, S] with unit stride along S
bool bhs(const Tensor& t, int64_t* batch_stride, int64_t* head_stride) {
  const auto n = t.sizes();
  const auto st = t.strides();
  if (n[2] != 1 && st[2] != 1) return false;
  *batch_stride = n[0] > 1 ? st[0] : n[1] * std::max(st[1], n[2]);
  *head_stride = n[1] > 1 ? st[1] : n[2];
  return true;
}

bool dtype_code(const Tensor& t, int32_t* code) {
  if (t.scalar_type() == at::kBFloat16) *code = PITH_BF16;
  else if (t.scalar_type() == at::kFloat) *code = PITH_F32;
  else return false;
  return true;
}

bool head_dims_ok(int64_t dq, int64_t dv) { return (dq == 64 && dv == 64) || (dq == 128 && dv == 128) || (dq == 192 && dv == 128); }

pith_stream_t stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor empty_like_shape(const Tensor& like, at::IntArrayRef shape, at::ScalarType dtype) {
  return at::empty(shape, like.options().dtype(dtype));
}

// ---------------------------------------------------------------------------------------------
// Chunk attention

// The shared rotary key part ([b, s, 64] or [b, s, 1, 64], unit stride along the features).
bool k_pe_fields(const Tensor& k, const Tensor& k_pe_in, const void** ptr, int64_t* bs, int64_t* rs) {
  Tensor pe = k_pe_in;
  if (pe.dim() == 4) {
    if (pe.size(2) != 1) return false;
    pe = pe.select(2, 0);
  }
  const int64_t b = k.size(0), s = k.size(1);
  if (!is_gpu_bf16(pe, 3) || pe.device() != k.device() || !has_shape(pe, {b, s, 64}) || pe.stride(2) != 1) return false;
  *rs = s > 1 ? pe.stride(1) : 64;
  *bs = b > 1 ? pe.stride(0) : s * *rs;
  *ptr = pe.data_ptr();
  return true;
}

// dtypes, shapes and devices of q, k, v (and k_pe) as the operators require them
bool qkv_ok(const Tensor& q, const Tensor& k, const Tensor& v, bool causal, bool two_part) {
  if (!is_gpu_bf16(q, 4) || !is_gpu_bf16(k, 4) || !is_gpu_bf16(v, 4) || k.device() != q.device() || v.device() != q.device()) return false;
  const int64_t dq = q.size(3), dv = v.size(3);
  if (!head_dims_ok(dq, dv) || k.size(3) != (two_part ? 128 : dq) || (two_part && (dq != 192 || q.size(2) != k.size(2)))) return false;
  if (k.size(0) != q.size(0) || v.size(0) != q.size(0) || k.size(1) != v.size(1) || k.size(2) != v.size(2)) return false;
  return k.size(2) > 0 && q.size(2) % k.size(2) == 0 && (!causal || q.size(1) == k.size(1));
}

using Rows = std::optional<std::pair<int64_t, int64_t>>;

// o, lse <- attention(q, k, v), see attn_fwd_into in operators/mla/hip.py. False: nothing was launched.
bool attn_fwd_into(const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& o, const Tensor& lse, double scale, bool causal,
                   const OptTensor& k_pe, const OptTensor& prev_o, const OptTensor& acc_o, const Rows& o_rows, const Rows& acc_o_rows) {
  if (!qkv_ok(q, k, v, causal, k_pe.has_value())) return false;
  const int64_t b = q.size(0), sq = q.size(1), hq = q.size(2), dv = v.size(3);
  const std::array<int64_t, 4> o_shape = {b, sq, hq, dv};
  pith_attn_fwd_args a = {};
  if (!is_gpu_f32(lse, 3) || lse.device() != q.device() || !has_shape(lse, {b, hq, sq}) || !bhs(lse, &a.lse_bs, &a.lse_hs)) return false;
  if (!bshd(q, &a.q_bs) || !bshd(k, &a.k_bs) || !bshd(v, &a.v_bs)) return false;
  if (o) {
    if (!is_gpu_bf16(*o, 4) || o->device() != q.device() || !has_shape(*o, o_shape) || !bshd(*o, &a.o_bs)) return false;
    a.o = o->data_ptr();
  }
  if (prev_o) {
    if (!prev_o->is_cuda() || prev_o->device() != q.device() || prev_o->dim() != 4 || !has_shape(*prev_o, o_shape) || (!o && !acc_o) ||
        !bshd(*prev_o, &a.prev_o_bs) || !dtype_code(*prev_o, &a.prev_o_dtype))
      return false;
    a.prev_o = prev_o->data_ptr();
    if (acc_o) {
      if (!is_gpu_f32(*acc_o, 4) || acc_o->device() != q.device() || !has_shape(*acc_o, o_shape) || !bshd(*acc_o, &a.acc_o_bs)) return false;
      a.acc_o = acc_o->data_ptr<float>();
    }
    if (o_rows) a.o_rows[0] = o_rows->first, a.o_rows[1] = o_rows->second;
    if (acc_o_rows) a.acc_o_rows[0] = acc_o_rows->first, a.acc_o_rows[1] = acc_o_rows->second;
  } else if (!o || acc_o) {
    return false;
  }
  if (k_pe && !k_pe_fields(k, *k_pe, &a.k_pe, &a.k_pe_bs, &a.k_pe_rs)) return false;
  a.q = q.data_ptr(); a.k = k.data_ptr(); a.v = v.data_ptr(); a.lse = lse.data_ptr<float>();
  a.B = b; a.Sq = sq; a.Skv = k.size(1); a.Hq = hq; a.Hkv = k.size(2); a.Dqk = q.size(3); a.Dv = dv;
  a.scale = (float)scale; a.causal = causal;
  return accepted(pith_attn_fwd(&a, stream_of(q)));
}

bool attn_bwd_delta_into(const Tensor& out, const Tensor& dout, const Tensor& delta) {
  if (!is_gpu_bf16(out, 4) || !is_gpu_bf16(dout, 4) || dout.device() != out.device() || dout.sizes() != out.sizes()) return false;
  pith_attn_delta_args a = {};
  a.B = out.size(0); a.S = out.size(1); a.H = out.size(2); a.D = out.size(3);
  if (!is_gpu_f32(delta, 3) || delta.device() != out.device() || !has_shape(delta, {a.B, a.H, a.S}) || !bhs(delta, &a.delta_bs, &a.delta_hs) ||
      !bshd(out, &a.o_bs) || !bshd(dout, &a.dout_bs))
    return false;
  a.o = out.data_ptr(); a.dout = dout.data_ptr(); a.delta = delta.data_ptr<float>();
  return accepted(pith_attn_bwd_delta(&a, stream_of(out)));
}

// What both backward calls of a chunk pair share.
bool bwd_args(pith_attn_bwd_args& a, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& dout, const Tensor& lse, const Tensor& delta,
              double scale, bool causal, const OptTensor& k_pe, const OptTensor& ds) {
  if (!qkv_ok(q, k, v, causal, k_pe.has_value())) return false;
  const int64_t b = q.size(0), sq = q.size(1), hq = q.size(2), hkv = k.size(2), dv = v.size(3);
  if (!is_gpu_bf16(dout, 4) || dout.device() != q.device() || !has_shape(dout, {b, sq, hq, dv})) return false;
  int64_t d_bs, d_hs, do_rh, v_rh;
  for (const Tensor* t : {&lse, &delta})
    if (!is_gpu_f32(*t, 3) || t->device() != q.device() || !has_shape(*t, {b, hq, sq})) return false;
  if (!bhs(lse, &a.lse_bs, &a.lse_hs) || !bhs(delta, &d_bs, &d_hs) || d_bs != a.lse_bs || d_hs != a.lse_hs) return false;
  if (!bshd_heads(q, &a.q_bs, &a.q_row_heads) || !bshd_heads(dout, &a.dout_bs, &do_rh) || !bshd_heads(k, &a.k_bs, &a.kv_row_heads) ||
      !bshd_heads(v, &a.v_bs, &v_rh) || do_rh != a.q_row_heads || v_rh != a.kv_row_heads)
    return false;
  if (k_pe && (a.q_row_heads != hq || a.kv_row_heads != hkv || !k_pe_fields(k, *k_pe, &a.k_pe, &a.k_pe_bs, &a.k_pe_rs))) return false;
  if (ds) {
    if (!ds->is_cuda() || ds->device() != q.device() || ds->scalar_type() != at::kByte || !ds->is_contiguous() || (uintptr_t)ds->data_ptr() % 256) return false;
    a.ds = ds->data_ptr();
    a.ds_bytes = ds->numel();
  }
  a.q = q.data_ptr(); a.k = k.data_ptr(); a.v = v.data_ptr(); a.dout = dout.data_ptr();
  a.lse = lse.data_ptr<float>(); a.delta = delta.data_ptr<float>();
  a.B = b; a.Sq = sq; a.Skv = k.size(1); a.Hq = hq; a.Hkv = hkv; a.Dqk = q.size(3); a.Dv = dv;
  a.scale = (float)scale; a.causal = causal;
  a.dq_dtype = a.dkv_dtype = PITH_BF16;
  return true;
}

// dK/dV side of a backward call: outputs and, in `workspace`, the scratch (stream order keeps the block alive until the
// kernels that use it have run).
bool dkdv_args(pith_attn_bwd_args& a, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& dk, const Tensor& dv, bool accumulate,
               const OptTensor& k_pe, const OptTensor& dk_pe, int64_t zero_tail, Tensor& workspace) {
  if (!dk.is_cuda() || dk.device() != q.device() || dv.device() != q.device() || dk.sizes() != k.sizes() || dv.sizes() != v.sizes() ||
      dk.scalar_type() != dv.scalar_type() || !dtype_code(dk, &a.dkv_dtype))
    return false;
  if (k_pe) {
    const int64_t b = k.size(0), s = k.size(1);
    if (!dk_pe || !dk_pe->is_cuda() || dk_pe->device() != q.device() || !has_shape(*dk_pe, {b, s, 64}) || dk_pe->scalar_type() != dk.scalar_type() ||
        dk_pe->stride(2) != 1 || (s > 1 && dk_pe->stride(1) != 64))
      return false;
    a.dk_pe = dk_pe->data_ptr();
    a.dk_pe_bs = b > 1 ? dk_pe->stride(0) : s * 64;
  }
  int64_t dk_rh, dv_rh;
  if (!bshd_heads(dk, &a.dk_bs, &dk_rh) || !bshd_heads(dv, &a.dv_bs, &dv_rh) || dk_rh != a.kv_row_heads || dv_rh != a.kv_row_heads) return false;
  a.dk = dk.data_ptr(); a.dv = dv.data_ptr();
  a.accumulate_dkv = accumulate;
  a.dkv_zero_tail = zero_tail;
  const int64_t need = pith_attn_bwd_dkdv_workspace_bytes(&a);
  if (need > 0) {
    workspace = empty_like_shape(q, {need}, at::kByte);
    a.workspace = workspace.data_ptr();
    a.workspace_bytes = need;
  }
  return true;
}

bool dq_args(pith_attn_bwd_args& a, const Tensor& q, const Tensor& dq, bool accumulate, const OptTensor& dq_final, const Rows& dq_final_rows) {
  int64_t rh;
  if (!dq.is_cuda() || dq.device() != q.device() || dq.sizes() != q.sizes() || !dtype_code(dq, &a.dq_dtype) || !bshd_heads(dq, &a.dq_bs, &rh) ||
      rh != a.q_row_heads)
    return false;
  a.dq = dq.data_ptr();
  a.accumulate_dq = accumulate;
  if (dq_final) {
    if (!is_gpu_bf16(*dq_final, 4) || dq_final->device() != q.device() || dq_final->sizes() != q.sizes() ||
        !bshd_heads(*dq_final, &a.dq_final_bs, &rh) || rh != a.q_row_heads)
      return false;
    a.dq_final = dq_final->data_ptr();
    if (dq_final_rows) a.dq_final_rows[0] = dq_final_rows->first, a.dq_final_rows[1] = dq_final_rows->second;
  }
  return true;
}

bool attn_bwd_dkdv_into(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& dout, const Tensor& lse, const Tensor& delta, const Tensor& dk,
                        const Tensor& dv, double scale, bool causal, bool accumulate, const OptTensor& k_pe, const OptTensor& dk_pe,
                        const OptTensor& ds, int64_t zero_tail) {
  pith_attn_bwd_args a = {};
  Tensor workspace;
  return bwd_args(a, q, k, v, dout, lse, delta, scale, causal, k_pe, ds) && dkdv_args(a, q, k, v, dk, dv, accumulate, k_pe, dk_pe, zero_tail, workspace) &&
         accepted(pith_attn_bwd_dkdv(&a, stream_of(q)));
}

bool attn_bwd_dq_into(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& dout, const Tensor& lse, const Tensor& delta, const Tensor& dq,
                      double scale, bool causal, bool accumulate, const OptTensor& k_pe, const OptTensor& ds, const OptTensor& dq_final,
                      const Rows& dq_final_rows) {
  pith_attn_bwd_args a = {};
  return bwd_args(a, q, k, v, dout, lse, delta, scale, causal, k_pe, ds) && dq_args(a, q, dq, accumulate, dq_final, dq_final_rows) &&
         accepted(pith_attn_bwd_dq(&a, stream_of(q)));
}

// Both of them; `ds` is the hand-over buffer between the two, if any.
bool attn_bwd_pair_into(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& dout, const Tensor& lse, const Tensor& delta, const Tensor& dq,
                        const Tensor& dk, const Tensor& dv, double scale, bool causal, bool accumulate_dq, bool accumulate_dkv, const OptTensor& k_pe,
                        const OptTensor& dk_pe, const OptTensor& ds, int64_t zero_tail, const OptTensor& dq_final, const Rows& dq_final_rows) {
  pith_attn_bwd_args a = {};
  Tensor workspace;
  return bwd_args(a, q, k, v, dout, lse, delta, scale, causal, k_pe, ds) &&
         dkdv_args(a, q, k, v, dk, dv, accumulate_dkv, k_pe, dk_pe, zero_tail, workspace) && dq_args(a, q, dq, accumulate_dq, dq_final, dq_final_rows) &&
         accepted(pith_attn_bwd(&a, stream_of(q)));
}

// ---------------------------------------------------------------------------------------------
// One rank's ring share with all of its chunks at hand (operators/ring_attention/local.py): every chunk in one launch.

struct RingChunks {
  std::vector<pith_key_chunk> chunk;  // as pith_attn_fwd_chunks wants them: the own chunk, under the mask, last
  std::vector<int64_t> rank;          // owner of each
};

// The chunks rank `rank` of `cp` visits, in ring order, and in `a` what they share. False: not a case for the chunk calls.
template <typename Args>
bool ring_chunks(const Tensor& q, const std::vector<OptTensor>& ks, const std::vector<OptTensor>& vs, const std::optional<std::vector<OptTensor>>& pes,
                 int64_t rank, int64_t cp, bool zigzag, Args& a, RingChunks& r) {
  if (!is_gpu_bf16(q, 4) || !q.is_contiguous() || rank < 0 || rank >= cp || (int64_t)ks.size() != cp || (int64_t)vs.size() != cp || (pes && (int64_t)pes->size() != cp))
    return false;
  const int64_t s = q.size(1);
  if (zigzag && s % 2) return false;
  for (int64_t step = 1; step <= cp; ++step) {
    const int64_t j = (rank - step + cp) % cp;  // the own chunk comes last
    if (!zigzag && j > rank) continue;
    if (!ks[j] || !vs[j] || (pes && !(*pes)[j])) return false;
    const Tensor &k = *ks[j], &v = *vs[j];
    if (!qkv_ok(q, k, v, true, pes.has_value()) || !k.is_contiguous() || !v.is_contiguous() || k.size(2) != ks[rank]->size(2)) return false;
    pith_key_chunk c = {};
    c.k = k.data_ptr(); c.v = v.data_ptr();
    c.rows = zigzag && j < rank ? s / 2 : s;
    c.q_row0 = j > rank ? s / 2 : 0;
    c.zero_tail = s - c.rows;
    int64_t pe_bs = 0, pe_rs = 0;
    if (pes && !k_pe_fields(k, *(*pes)[j], &c.k_pe, &pe_bs, &pe_rs)) return false;
    if (!r.chunk.empty() && (pe_bs != a.k_pe_bs || pe_rs != a.k_pe_rs)) return false;
    a.k_pe_bs = pe_bs; a.k_pe_rs = pe_rs;
    r.chunk.push_back(c);
    r.rank.push_back(j);
  }
  if (r.chunk.size() > PITH_MAX_CHUNKS) return false;
  const Tensor &k = *ks[rank], &v = *vs[rank];
  a.q = q.data_ptr();
  a.B = q.size(0); a.Sq = s; a.Hq = q.size(2); a.Hkv = k.size(2); a.Dqk = q.size(3); a.Dv = v.size(3);
  a.q_bs = s * a.Hq * a.Dqk; a.k_bs = s * a.Hkv * k.size(3); a.v_bs = s * a.Hkv * a.Dv;
  a.lse_bs = a.Hq * s; a.lse_hs = s;
  a.causal = 1;
  return true;
}

// Compute units of a device, looked up once.
int64_t compute_units(int device) {
  static std::array<std::atomic<int>, 64> cached = {};
  if (device < 0 || device >= 64) return 0;
  int n = cached[device].load(std::memory_order_relaxed);
  if (n == 0) {
    pith_device_info_t info;
    if (pith_device_info(device, &info) != PITH_OK) return 0;
    cached[device].store(n = info.compute_units, std::memory_order_relaxed);
  }
  return n;
}

// Whether a share's forward goes out as one launch over its chunks, or as one launch per ring step. One launch saves launches
// and merges; but its loop keeps the state of several walks, and one work split has to serve chunks with and without a mask,
// where the steps take the best for each. That shows where workgroups are few and streams long. rows = query rows, wgs = 128-row
// workgroups, mean = mean length of the rows' streams in percent of the longest. One launch against steps, time ratio:
//   more than two workgroups per compute unit, or 64-row ones fit:  0.85-1.01
//   up to two    8192 x 8 heads of 128, mean 50 / 57 / 67 / 75      1.00 / 1.02 / 1.07 / 1.07      16384 x 4  1.04 / 1.06 / 1.09 / 1.10
//                16384 x 4 of 192 1.04 / 1.06 / 1.06 / 1.07         8192 x 8  1.00 / 1.01 / 1.03 / 1.03
//                3072 x 16 of 128 0.90 / 0.87 / 0.98 / 1.04         4096 x 16 of 192  0.95 / 0.94 / 0.98 / 1.00
//   up to one    8192 x 4 of 128  0.92 / 0.96 / 1.03 / 1.08         6144 x 4 of 192  0.91 / 0.88 / 1.03 / 1.14
//                16384 x 2 of 128 0.97 / 1.03 / 1.09 / 1.13         12288 x 2 of 192  0.99 / 0.94 / 1.06 / 1.22
//   two chunks only: 6144 x 8 of 128 1.04 (mean 50), 1.10 (75); eight chunks: 8192 x 8 of 192 0.96, 16384 x 4 1.06
bool share_forward_in_one(int64_t dqk, int64_t rows, int64_t heads, int64_t chunks, int64_t mean, int64_t cus) {
  const int64_t wgs = (rows + 127) / 128 * heads, wgs64 = (rows + 63) / 64 * heads;
  if (dqk == 64 || chunks == 1 || wgs > 2 * cus || wgs64 <= cus) return true;
  if (rows >= 12288 || (rows >= 8192 && chunks < 8)) return wgs <= cus && mean <= 60;
  if (wgs <= cus) return rows < 6144 || mean <= 65;
  return !(chunks == 2 && (rows >= 6144 || (dqk == 128 && mean > 70 && rows >= 3072)));
}

// (out, lse), or None when the steps have to run one by one.
std::optional<std::tuple<Tensor, Tensor>> ring_forward(const Tensor& q, const std::vector<OptTensor>& ks, const std::vector<OptTensor>& vs,
                                                       const std::optional<std::vector<OptTensor>>& pes, double scale, int64_t rank, int64_t cp,
                                                       bool zigzag) {
  pith_attn_fwd_args a = {};
  RingChunks r;
  if (!ring_chunks(q, ks, vs, pes, rank, cp, zigzag, a, r)) return std::nullopt;
  int64_t keys = 0, seen = 0;  // in the chunks; (query row, key) pairs
  for (const pith_key_chunk& c : r.chunk) {
    keys += c.rows;
    seen += &c == &r.chunk.back() ? c.rows * a.Sq / 2 : c.rows * (a.Sq - c.q_row0);
  }
  if (keys * a.Sq > 0 && !share_forward_in_one(a.Dqk, a.Sq, a.Hq * a.B, (int64_t)r.chunk.size(), 100 * seen / (keys * a.Sq), compute_units(q.device().index())))
    return std::nullopt;
  Tensor o = at::empty({a.B, a.Sq, a.Hq, a.Dv}, q.options());
  Tensor lse = empty_like_shape(q, {a.B, a.Hq, a.Sq}, at::kFloat);
  a.o = o.data_ptr(); a.lse = lse.data_ptr<float>();
  a.o_bs = a.Sq * a.Hq * a.Dv;
  a.scale = (float)scale;
  if (!accepted(pith_attn_fwd_chunks(&a, r.chunk.data(), (int64_t)r.chunk.size(), stream_of(q)))) return std::nullopt;
  return std::make_tuple(o, lse);
}

// The same for the backward without a dS hand-over. One grid over all chunks fills the rounds that a step's kernels leave half
// empty; long streams of whole chunks whose query workgroups come in whole rounds have none, and a step can cut the heads of
// its chunk finer. One grid against steps, 128 features: 8192 x 8/2 heads, 4 ranks 1850 and 1744 us (rank 0), 8 ranks,
// contiguous 3790 and 3480, 16384 x 8/2, 2 ranks 3320 and 3130, 16384 x 4 contiguous 5464 and 5377; but 9216 x 8/2, 8 ranks
// 4593 and 4746, 12288 x 8/2 rank 0 3736 and 3675, rank 1 (half chunks) 3594 and 3747, 8192 x 8/2 rank 1 1705 and 1738.
// Beyond the one grid (two launches; a share of that size recomputes only for want of memory) the same holds of half chunks
// too: 8192 x 32/4 6707 and 6202, rank 1 6702 and 6249, 4096 x 64/4 3715 and 3246, but 6144 x 32/4 rank 3 3574 and 3864.
bool share_backward_in_one(int64_t dqk, int64_t rows, int64_t heads, int64_t chunks, int64_t keys, int64_t cus) {
  const int64_t wgs = (rows + 127) / 128 * heads;
  if (dqk != 128 || chunks == 1 || cus == 0) return true;
  if (wgs > 4 * cus) return rows < 4096 || wgs % (4 * cus) != 0;
  return rows < 8192 || keys < chunks * rows || wgs % (2 * cus) != 0;
}

// Bytes of the buffer through which a share's one dK/dV launch hands dS to its one dQ launch, 0 where it recomputes.
// Against one grid of both kinds (two recomputing launches from W 1 on) that loses the last round of either launch and wins two products
// of seven. W = its 256-row dQ workgroups per compute unit; backward, handing over / recomputing, us, four ranks unless named, zigzag rank 1
// and contiguous rank 1:
//   W 0.25  1024 x 16 123 / 88 and 143 / 106               W 0.5   2048 x 16 300 / 287 and 224 / 216, 8192 x 4 1077 / 1055 and 800 / 788, 4 x 512 x 16 110 / 101
//   W 0.75  3072 x 16 567 / 640 and 679 / 777, 12032 x 4 2055 / 2326 and 2466 / 2873, 2 x 1536 x 16 313 / 349 and 361 / 418
//   W 1     4096 x 16 948 / 1052 and 678 / 790, 8 ranks 1825 / 2066 and 2444 / 2801, 2 x 2048 x 16 519 / 568 and 361 / 422, 4 x 1024 x 16 310 / 336 and
//           209 / 244, 16384 x 4 3575 / 4007 and 2630 / 3008    W 1.25-2   5120 x 16, 2 ranks 740 / 838, 6144 x 16 2054 / 2322, 8192 x 16, 2 ranks 1776 / 2017
// Keys in two parts the same: 4096 x 16 969 / 1063, 4 x 1024 x 16 316 / 344. Rows below 1024 gain on the device as well, W 1-2, zigzag and contiguous: 4 x
// 896 x 16 257 / 280 and 180 / 203, 8 x 640 x 16 295 / 321 and 207 / 233, 8 x 512 x 16 212 / 225 and 146 / 165, 512 x 128 213 / 226 and 152 / 170 (16 x 256 x 16
// zigzag loses, 194 / 190). The line was drawn before these were measured and has not been weighed against the host: the Python body, which owns the
// buffer, takes 136 us of its time, the native one 108, about as long as the shorter of these kernels. A zigzag share whose half chunk is no multiple of 64 rows has no such hand-over (a 64-row tile would
// lie across two images, pith_attn_bwd_chunks_ds_bytes) and pays 13 % of its backward: 4160 x 16 1198, recomputing, where 4224 x 16 takes
// 1040 (1220 recomputing); 6146 x 16 2355 beside 1988 for 6144, 2 x 2050 x 16 660 beside 508 for 2 x 2048 (both with a further round).
bool share_of_192_pays(int64_t b, int64_t rows, int64_t hq, int64_t cus) { return cus > 0 && rows >= 1024 && 10 * ((rows + 255) / 256 * hq * b) >= 7 * cus; }
int64_t share_ds_bytes(const Tensor& q, const std::vector<OptTensor>& ks, const std::vector<OptTensor>& vs, const std::optional<std::vector<OptTensor>>& pes,
                       int64_t rank, int64_t cp, bool zigzag) {
  if (!q.is_cuda() || q.dim() != 4 || q.size(3) != 192 || !share_of_192_pays(q.size(0), q.size(1), q.size(2), compute_units(q.device().index()))) return 0;
  pith_attn_bwd_args a = {};
  RingChunks r;
  return ring_chunks(q, ks, vs, pes, rank, cp, zigzag, a, r) ? pith_attn_bwd_chunks_ds_bytes(&a, r.chunk.data(), (int64_t)r.chunk.size()) : 0;
}

// (dq, dk list, dv list, dk_pe list or empty); the lists hold a tensor per visited chunk. None as above. The policy for the
// dS hand-over is the caller's: without its buffer of share_ds_bytes this call recomputes.
using RingGrads = std::tuple<Tensor, std::vector<OptTensor>, std::vector<OptTensor>, std::vector<OptTensor>>;
std::optional<RingGrads> ring_backward(const Tensor& dout_in, const Tensor& q, const Tensor& out, const Tensor& lse, const std::vector<OptTensor>& ks,
                                       const std::vector<OptTensor>& vs, const std::optional<std::vector<OptTensor>>& pes, double scale, int64_t rank,
                                       int64_t cp, bool zigzag, const OptTensor& ds) {
  pith_attn_bwd_args a = {};
  RingChunks r;
  if (!ring_chunks(q, ks, vs, pes, rank, cp, zigzag, a, r)) return std::nullopt;
  int64_t keys = 0;
  for (const pith_key_chunk& c : r.chunk) keys += c.rows;
  if (!share_backward_in_one(a.Dqk, a.Sq, a.Hq * a.B, (int64_t)r.chunk.size(), keys, compute_units(q.device().index()))) return std::nullopt;
  if (!is_gpu_bf16(dout_in, 4) || !is_gpu_bf16(out, 4) || !out.is_contiguous() || !is_gpu_f32(lse, 3) || !lse.is_contiguous() ||
      dout_in.device() != q.device() || out.device() != q.device() || lse.device() != q.device() || !has_shape(dout_in, {a.B, a.Sq, a.Hq, a.Dv}) ||
      !has_shape(out, {a.B, a.Sq, a.Hq, a.Dv}) || !has_shape(lse, {a.B, a.Hq, a.Sq}))
    return std::nullopt;
  const Tensor dout = dout_in.contiguous();
  Tensor delta = empty_like_shape(q, {a.B, a.Hq, a.Sq}, at::kFloat), dq = at::empty_like(q), workspace;
  if (!attn_bwd_delta_into(out, dout, delta)) return std::nullopt;
  a.dout = dout.data_ptr(); a.lse = lse.data_ptr<float>(); a.delta = delta.data_ptr<float>(); a.dq = dq.data_ptr();
  a.dout_bs = a.Sq * a.Hq * a.Dv;
  a.dq_bs = a.q_bs; a.dk_bs = a.k_bs; a.dv_bs = a.v_bs;
  a.dk_pe_bs = a.Sq * 64;
  a.dq_dtype = a.dkv_dtype = PITH_BF16;
  a.scale = (float)scale;
  if (ds && (!ds->is_cuda() || ds->device() != q.device() || ds->scalar_type() != at::kByte || !ds->is_contiguous() || (uintptr_t)ds->data_ptr() % 256)) return std::nullopt;
  RingGrads g = {dq, std::vector<OptTensor>(cp), std::vector<OptTensor>(cp), std::vector<OptTensor>(pes ? cp : 0)};
  for (size_t i = 0; i < r.chunk.size(); ++i) {
    const int64_t j = r.rank[i];
    Tensor dk = at::empty_like(*ks[j]), dv = at::empty_like(*vs[j]);
    r.chunk[i].dk = dk.data_ptr(); r.chunk[i].dv = dv.data_ptr();
    std::get<1>(g)[j] = dk;
    std::get<2>(g)[j] = dv;
    if (pes) {
      Tensor dk_pe = at::empty({a.B, a.Sq, 64}, q.options());
      r.chunk[i].dk_pe = dk_pe.data_ptr();
      std::get<3>(g)[j] = dk_pe;
    }
  }
  const int64_t n = (int64_t)r.chunk.size(), need = pith_attn_bwd_chunks_workspace_bytes(&a, r.chunk.data(), n);
  if (need > 0) {
    workspace = empty_like_shape(q, {need}, at::kByte);
    a.workspace = workspace.data_ptr();
    a.workspace_bytes = need;
  }
  if (!accepted(pith_attn_bwd_chunks_handover(&a, r.chunk.data(), n, ds ? ds->data_ptr() : nullptr, ds ? ds->numel() : 0, stream_of(q)))) return std::nullopt;
  return g;
}

using Two = std::tuple<Tensor, Tensor>;
using Three = std::tuple<Tensor, Tensor, Tensor>;
using Four = std::tuple<Tensor, Tensor, Tensor, Tensor>;

Two attn_fwd(const Tensor& q, const Tensor& k, const Tensor& v, double scale, bool causal) {
  if (q.is_cuda() && q.dim() == 4 && v.dim() == 4) {
    Tensor o = at::empty({q.size(0), q.size(1), q.size(2), v.size(3)}, q.options().dtype(at::kBFloat16));
    Tensor lse = at::empty({q.size(0), q.size(2), q.size(1)}, q.options().dtype(at::kFloat));
    if (attn_fwd_into(q, k, v, o, lse, scale, causal, {}, {}, {}, {}, {})) return {o, lse};
  }
  return python_body<Two>("attn_fwd", q, k, v, scale, causal);
}

// Whether a dQ kernel that reads handed-over dS (512 query rows per workgroup) beats recomputing the scores: it has to fill the
// device, or two thirds of it with rows. By those rows in 512 per compute unit, forward + backward, handing over / recomputing, us (to 16384 rows):
//   causal  0.5-0.65   2100 x 32/4 heads 214 / 193, 3 x 768 x 32/4 117 / 105, 2 x 1200 x 32/4 151 / 144, 2 x 1300 x 32/4 168 / 164, 2500 x 32/4 264 / 270, 5 x 512 x 32
//                      112 / 107, 5 x 1000 x 16/4 138 / 137    0.68   7 x 400 x 32/4 119 / 116
//           0.69-0.75  2816 x 32/4 305 / 318, 3 x 1900 x 16 219 / 229, 3 x 960 x 32/4 140 / 147, 3000 x 32/4 335 / 357, 1500 x 64/4 194 / 202, 6000 x 16 588 / 615
//           0.8-0.95   13 x 512 x 16 131 / 139, 7 x 500 x 32/4 132 / 139, 13000 x 8/2 1298 / 1396, 3500 x 32/4 415 / 445, 7 x 1024 x 16 182 / 193, 15000 x 8/2 1644 / 1795
//   full    0.69-0.75  3 x 1900 x 16 376 / 404, 3 x 1000 x 32/4 231 / 237, 1500 x 64/4 325 / 342, 6000 x 16 1067 / 1173
//           0.8-0.95   13 x 512 x 16 160 / 179, 3500 x 32/4 772 / 829, 7 x 512 x 32/4 155 / 167, 15000 x 8/2 3202 / 3478
// From a full device on, W = workgroups per compute unit; forward + backward, inputs changing, handing over / recomputing, us:
//   causal  W 1     4096 x 32/4 heads 561 / 576, 8192 x 16 1030 / 1059, 2 x 2048 x 32/4 323 / 332, 4 x 1024 x 32/4 204 / 215, 8 x 512 x 32/4 148 / 162
//           W 1.12  9216 x 16 1378 / 1392, 3 x 1536 x 32/4 305 / 312, 9 x 512 x 32/4 189 / 190
//           W 1.25  5120 x 32/4 891 / 914, 2 x 2560 x 32/4 496 / 502       W 1.5   6144 x 32/4 1229 / 1265, 6 x 1024 x 32/4 310 / 317,
//                   3 x 1999 x 32/4 487 / 500, 2 x 3072 x 32/4 677 / 693   W 1.75  7168 x 32/4 1600 / 1651
//           W 2     8192 x 32/4 2055 / 2103, 16 x 512 x 32/4 262 / 276     W 2.25  9216 x 32/4 2611 / 2721, 9 x 1024 x 32/4 443 / 461
//           W 3     12288 x 32/4 4524 / 4756                               W 4     16384 x 32/4 7929 / 8004, 16 x 1024 x 32/4 718 / 736
//   full    W 1     2 x 2048 x 32/4 534 / 539    W 1.12  4608 x 32/4 1625 / 1670, 9216 x 16 2716 / 2798
//           W 1.25  5120 x 32/4 1833 / 1887      W 1.5   6144 x 32/4 2367 / 2426
// And dK/dV, whose stores wait for memory, must not leave units idle that the recomputing dQ of one grid would take: a group
// of an odd number of heads is not split, and a slab of few heads is a small grid. F = its 128-key workgroups per unit; backward
// alone, causal and full unless one is named:
//   F 0.25-0.5  2 x 1536 x 44/4 452 / 430 and 550 / 518, 8 x 512 x 33/3 198 / 184 and 216 / 198, 4096 x 33/3 causal 1111 / 1057, 2048 x 36/4 x 2
//               505 / 485 and 639 / 612, 12288 x 11/1 3238 / 3084 and 3916 / 3863, 4096 x 76/4 1964 / 1947 and 2432 / 2353, 4096 x 52/4 0-1 % slower;
//               8192 x 4096 in slabs, full: 66/6 in two 5452 / 3615, 88/8 in two 5636 / 4428
//   F 0.62      4096 x 35/5 causal 786 / 776, 2 x 2048 x 35/5 full 575 / 547, 4096 x 55/5 1191 / 1200 and 1612 / 1597
//   F 0.75      4096 x 66/6 1256 / 1282 and 1796 / 1868, 4 x 1536 x 44/4 528 / 536 and 718 / 726, 2 x 3072 x 44/4 causal 957 / 978
//   F 0.85      2 x 1536 x 45/9 275 / 274 and 384 / 387, 2 x 2048 x 35/7 344 / 345 and 498 / 510
//   F 1, 1.4    4096 x 40/8 causal 666 / 690, 2 x 2048 x 33/11 282 / 284 and 508 / 549
// And few workgroups may be mostly empty:
//   up to 256 rows         8 x 64 x 32/4 51 / 29 and 44 / 35 (64/4 heads), 8 x 128 x 32/4 48 / 39 and 44 / 38, 64 x 64 x 32/4 113 / 91 and 91 / 70, 1024 x
//                          100 x 4/1 258 / 220, 32 x 192 x 8 49.2 / 48.5 and 52.4 / 52.1, 8 x 256 x 32/4 76 / 74 and 65 / 64, 64 x 256 x 16/4 158 / 159 and
//                          175 / 179 (and such calls spend more time in Python than on the device)
//   257 to 512             8 x 257 x 32/4 90 / 94 and 88 / 91, 32 x 320 x 8 78 / 84 and 92 / 101, 64 x 384 x 16/4 257 / 264 and 319 / 340; worst 16 x 288 x 32/4
//                          full 157 / 155
//   full, 513 to 639 rows  4 x 513 x 32/4 127 / 108, 4 x 600 x 32/4 138 / 119, 4 x 513 x 64/4 222 / 211, 16 x 540 x 32/4 410 / 391, 8 x 600 x 16 129 / 123;
//                          640 and more 8 x 640 x 32/8 232 / 233, 16 x 640 x 32/4 439 / 441, 8 x 720 x 16 155 / 164
//   causal, from 513 on    4 x 513 x 32/4 98 / 99, 4 x 600 x 32/4 113 / 110, 8 x 600 x 32/4 167 / 173, 4 x 600 x 64/4 168 / 174, 8 x 1025 x 32/4 333 / 354
bool ds_handover_pays(int64_t b, int64_t sq, int64_t skv, int64_t hq, int64_t hkv, bool causal, int64_t cus) {
  if (cus <= 0 || !pith::handover_rows_pay(b, sq, hq, causal, cus)) return false;
  pith_attn_bwd_args a = {};
  a.B = b; a.Sq = sq; a.Skv = skv; a.Hq = hq; a.Hkv = hkv; a.Dqk = a.Dv = 128; a.causal = causal;
  pith_attn_bwd_plan_t plan;
  if (pith_attn_bwd_plan(&a, &plan) != PITH_OK) return false;
  const int64_t key_tiles = (skv + plan.dkdv_rows - 1) / plan.dkdv_rows * plan.dkdv_rows / 128;
  const int64_t dkdv_wgs = key_tiles * hkv * b * plan.dkdv_split;
  // (causal 7900 x 12/4, 248 of them: 887 / 837)
  if (causal && 2 * dkdv_wgs < 3 * cus && !pith::handover_fills_device(b, sq, hq, cus)) return false;
  return 4 * dkdv_wgs >= 3 * cus;
}

// The same for (192, 128): its dQ kernel takes 256 rows per workgroup.
// W = 256-row workgroups per compute unit, F as above; backward alone, inputs changing, handing over / recomputing, us (16 heads unless
// others are named):
//   causal  W 0.5         2048 104 / 88, 1024 x 32 61 / 52, 8192 x 4 336 / 287    W 0.75  3072 156 / 170, 12288 x 4 581 / 610, 3 x 1021 69 / 82
//           W 1           4096 243 / 282, 2 x 2048 135 / 161, 4 x 1024 82 / 98, 8 x 512 60 / 66, 512 x 128 59 / 65, 16384 x 4 917 / 1036, 4096 x 16/4 265 / 301
//           W 1.12-2.25   4608 326 / 379, 5120 396 / 454, 6144 542 / 614, 3 x 1999 204 / 229, 7168 706 / 790, 1024 x 128 171 / 189, 9216 1176 / 1308
//   full    F below 0.75  2048 x 1024 85 / 74, 8192 x 4096 x 4 292 / 268, 2731 x 1366 127 / 140    W 0.25  1024 x 2048 91 / 84, 4096 x 8192 x 4 313 / 290
//           W 0.5         2048 x 2048 128 / 139, 2 x 1024 x 2048 134 / 144, 8192 x 16384 x 4 942 / 994
//           W 0.6-1.25    2560 x 5120 391 / 428, 3072 x 1536 138 / 155, 3072 x 6144 507 / 604, 2 x 2048 x 1024 117 / 139, 5120 x 2560 426 / 503
// Below 2^25 visible pairs of rows and heads the device gains as much, but the Python body of such a call takes longer than its kernels, on the
// host of one machine: forward + backward with the host's time 8 x 512 causal 93-120 / 102, 512 x 128 99-123 / 111; 4 x 1024 127 / 140.
bool ds_handover_pays_192(int64_t b, int64_t sq, int64_t skv, int64_t hq, int64_t hkv, bool causal, int64_t cus) {
  if (cus <= 0 || b * hq * sq * skv < (int64_t)(causal ? 64 : 32) << 20 || 10 * ((sq + 255) / 256 * hq * b) < (causal ? 7 : 5) * cus) return false;
  pith_attn_bwd_args a = {};
  a.B = b; a.Sq = sq; a.Skv = skv; a.Hq = hq; a.Hkv = hkv; a.Dqk = 192; a.Dv = 128; a.causal = causal;
  pith_attn_bwd_plan_t plan;
  if (pith_attn_bwd_plan(&a, &plan) != PITH_OK) return false;
  return 4 * ((skv + 127) / 128) * hkv * b * plan.dkdv_split >= 3 * cus;
}

// Whether a share that could be one launch over all chunks goes out step by step instead, because steps hand dS over; `steps`:
// (rows, keys, causal, kv heads of a slab that hands over at once, 0: recomputes). A step is a grid of its own for either kernel, and the last
// round of each is lost, which one launch does not know; handing over saves a fifth of the time where the grids are whole rounds. L =
// rounds of the unmasked steps that hand over against what their workgroups would fill, 0.7 for dK/dV and 0.3 for dQ as their times are;
// backward, steps / one launch, four ranks, rank 2 zigzag and contiguous unless another is named, us:
//   L 1          4096 x 64/4 heads 3208 / 3262 and 3779 / 3923, 8192 x 16 3028 / 3209 and 3643 / 3865, 16384 x 8 5864 / 6309 and 7072 / 7493, 8000 x 32/4 5879 / 6432
//                and 6980 / 7797
//   L 1.05-1.2   7680 x 32/4 5544 / 5988 and 6683 / 7265, 7168 x 32/4 5048 / 5330 and 6066 / 6328, 2 x 7168 x 32/4 9665 / 9372 and 11836 / 11701, 8192 x 40/8
//                7793 / 7664 and 9775 / 9485, 6000 x 32 3645 / 3502 and 4216 / 4223
//   L 1.2-1.4    6144 x 64/4 7452 / 7585 and 9372 / 9466, 3 x 4096 x 32/4 5248 / 5169 and 6285 / 6453, 6144 x 32/4 3979 / 3883 and 4737 / 4352, 11264 x 32/4 12720 /
//                11931 and 15956 / 14840, 5632 x 64/8 6604 / 5941 and 8074 / 7450, 4 x 3000 x 32/4 4005 / 3511 and 4796 / 4330
//   L 1.4-1.8    9216 x 32/4 9779 / 8198 and 12376 / 9958, 10240 x 32/4 11186 / 9970 and 14109 / 12097, 5120 x 32/4 2860 / 2531 and 3594 / 3132, 4608 x 32/4
//                2500 / 2134 and 3201 / 2614, 4 x 1100 x 64/4 1592 / 1152 and 1780 / 1329
// With short rows the fp32 dQ and the launches of every step weigh more: L 1, 2 x 2048 x 64/4 1783 / 1774 and 2103 / 2130 (two ranks 880 / 987
// and 1292 / 1381), 2 x 2048 x 32/4 two ranks, rank 0 502 / 475, 8 x 1024 x 32/4 1058 / 904 and 1139 / 1095, 16 x 512 x 32/4 720 / 508 and 700 / 594. Where
// only the masked step hands over (it has no half-empty round): half of the work, two ranks, rank 0 8192 x 16 1535 / 1582, 6144 x 32/4 1913 /
// 1867, 1792 x 64/4 448 / 394; less of it, 12288 x 16/2 contiguous 9341 / 8613, 1792 x 64/4 four ranks, rank 0 832 / 715. One launch means two from
// four dQ workgroups per unit on, and where dQ, two workgroups to a unit, leaves its last round half empty, the steps are faster from a
// quarter of the work on: two ranks, rank 0 4352 x 32/4 1058 / 1183, 20480 x 8/2 4975 / 5452, 2560 x 64/4 720 / 748, four ranks 1413 / 1555, 5120 x 32/4 2629 /
// 3013, 2304 x 64/4 1231 / 1303, 2 x 2304 x 32 1253 / 1259; whole rounds 3072 x 64/4 1021 / 977, four ranks 2067 / 2031.
// 192 features are asked only where the share as a whole does not hand over (share_of_192_pays, images beyond the buffer's limit, half chunks
// off the 64-row grid). The limits are those of 128 features: wherever they choose the steps these are faster, and what they leave out is mostly
// even. 16 heads, four ranks, rank 2 zigzag and contiguous unless others are named:
//   chosen     8192 3510 / 3798 and 4298 / 4692, 10240 5738 / 5993 and 6823 / 7755, 16384 x 8 6743 / 7422 and 8350 / 9251, 9216 contiguous 5796 / 6460, 12288 in slabs
//              of 8 heads contiguous 9822 / 10598, 8192 x 64/4 in slabs of 2 kv heads 14300 / 16940, 16 x 2048 4907 / 5001 and 5994 / 6372, 8 x 3072 4715 / 4944 and
//              5589 / 6000; half chunks off the grid: 7170 2935 / 3125, 2 x 4098 x 32 4307 / 4485, 16 x 2050 5408 / 5567, 8 x 2306 3111 / 3142
//   left out   4098 1332 / 1115, 3074 703 / 670, 64 x 1024 7357 / 6247, 2560 x 32 950 / 840, 9216 4903 / 4971, 5122 1724 / 1766, 8194 4148 / 4198; two ranks, rank 0, 3074 368 /
//              342, 4098 604 / 622, 8194 1972 / 2270
bool share_hands_over(int64_t b, int64_t rows, int64_t hq, int64_t hkv, const std::vector<std::array<int64_t, 4>>& steps, int64_t cus, int64_t dqk) {
  if (cus <= 0 || hkv <= 0) return false;
  if (steps.size() == 1) return steps[0][3] != 0;  // a call like any other
  const auto lost = [&](int64_t wgs, int per_unit = 1) {
    const int64_t round = per_unit * cus;
    return (double)((wgs + round - 1) / round * round) / (double)wgs;
  };
  double all = 0, handed = 0, full = 0, full_lost = 0;
  for (const auto& [sq, skv, causal, heads] : steps) {
    const double work = (double)sq * (double)skv * (causal ? 0.5 : 1.0);
    all += work;
    // (the measured shares handed over in steps that fill the device)
    if (heads == 0 || (dqk == 128 && (sq + 511) / 512 * (hq / hkv * heads) * b < cus)) continue;
    handed += work;
    if (causal) continue;
    pith_attn_bwd_args a = {};
    a.B = b; a.Sq = sq; a.Skv = skv; a.Hq = hq / hkv * heads; a.Hkv = heads; a.Dqk = dqk; a.Dv = 128;
    pith_attn_bwd_plan_t plan;
    if (pith_attn_bwd_plan(&a, &plan) != PITH_OK) return false;
    full += work;
    const int64_t dq_rows = dqk == 192 ? 256 : 512;
    full_lost += work * (0.7 * lost((skv + plan.dkdv_rows - 1) / plan.dkdv_rows * heads * b * plan.dkdv_split) + 0.3 * lost((sq + dq_rows - 1) / dq_rows * a.Hq * b));
  }
  if (handed == 0) return false;
  const int64_t q_wgs = (rows + 127) / 128 * hq * b;
  if (full == 0 && q_wgs > 4 * cus && rows >= 2304 && 4 * handed >= all && lost(q_wgs, 2) >= 1.1) return true;
  if (2 * handed < all) return false;
  if (rows >= 4096) return full_lost < 1.2 * full || full == 0;
  return rows >= 2048 && handed == all && (rows + 511) / 512 * hq * b >= 2 * cus && full_lost <= 1.05 * full;
}

// Whether any step of a share of (192, 128) could hand dS over, by its grids: its own chunk under the mask, and of the others whole chunks
// (contiguous), half the keys of those in front and half the rows against those behind (zigzag).
bool step_of_192_hands_over(int64_t b, int64_t s, int64_t hq, int64_t hkv, int64_t rank, int64_t cp, bool zigzag, int64_t cus) {
  const auto pays = [&](int64_t rows, int64_t keys, bool causal) { return ds_handover_pays_192(b, rows, keys, hq, hkv, causal, cus); };
  if (pays(s, s, true)) return true;
  if (!zigzag) return rank > 0 && pays(s, s, false);
  return (rank > 0 && pays(s, s / 2, false)) || (rank < cp - 1 && pays(s / 2, s, false));
}

Three attn_bwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& lse, const Tensor& dout, double scale, bool causal) {
  // Calls large enough for the dS hand-over belong to the Python body, which owns the policy for the hand-over buffer: their
  // kernels outlast its host work many times over.
  bool small = q.is_cuda() && q.dim() == 4 && v.dim() == 4;
  if (small && (q.size(3) == 128 || q.size(3) == 192) && k.dim() == 4) {
    const auto pays = q.size(3) == 128 ? ds_handover_pays : ds_handover_pays_192;
    small = !pays(q.size(0), q.size(1), k.size(1), q.size(2), k.size(2), causal, compute_units(q.device().index()));
  }
  if (small && q.is_contiguous() && k.is_contiguous() && v.is_contiguous()) {
    Tensor delta = empty_like_shape(q, {q.size(0), q.size(2), q.size(1)}, at::kFloat);
    Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    if (attn_bwd_delta_into(o, dout, delta) &&
        attn_bwd_pair_into(q, k, v, dout, lse, delta, dq, dk, dv, scale, causal, false, false, {}, {}, {}, 0, {}, {}))
      return {dq, dk, dv};
  }
  return python_body<Three>("attn_bwd", q, k, v, o, lse, dout, scale, causal);
}

// ---------------------------------------------------------------------------------------------
// Combine

bool combine_into(const Tensor& out1, const Tensor& lse1, const Tensor& out2, const Tensor& lse2, const Tensor& out, const Tensor& lse_out, int64_t base) {
  pith_combine_args a = {};
  if (!out1.is_cuda() || out1.dim() != 4) return false;
  for (const Tensor* t : {&out2, &out})
    if (t->device() != out1.device() || t->sizes() != out1.sizes()) return false;
  a.B = out1.size(0); a.S = out1.size(1); a.H = out1.size(2); a.D = out1.size(3);
  for (const Tensor* t : {&lse1, &lse2, &lse_out})
    if (!is_gpu_f32(*t, 3) || t->device() != out1.device() || !has_shape(*t, {a.B, a.H, a.S})) return false;
  if (!bhs(lse1, &a.lse1_bs, &a.lse1_hs) || !bhs(lse2, &a.lse2_bs, &a.lse2_hs) || !bhs(lse_out, &a.lse_out_bs, &a.lse_out_hs)) return false;
  if (!dtype_code(out1, &a.dtype1) || !dtype_code(out2, &a.dtype2) || !dtype_code(out, &a.dtype_out)) return false;
  if (!bshd(out1, &a.out1_bs) || !bshd(out2, &a.out2_bs) || !bshd(out, &a.out_bs)) return false;
  a.out1 = out1.data_ptr(); a.out2 = out2.data_ptr(); a.out = out.data_ptr();
  a.lse1 = lse1.data_ptr<float>(); a.lse2 = lse2.data_ptr<float>(); a.lse_out = lse_out.data_ptr<float>();
  a.base = (int32_t)base;
  return accepted(pith_combine(&a, stream_of(out1)));
}

// The reference's calling convention: fresh fp32 outputs. None when the Python body has to take the call.
std::optional<Two> combine_new(const Tensor& out1, const Tensor& lse1, const Tensor& out2, const Tensor& lse2, int64_t base) {
  if (!out1.is_cuda() || !lse1.is_cuda() || out1.dim() != 4 || lse1.dim() != 3 || (!lse1.is_contiguous() && lse1.stride(-1) != 1)) return std::nullopt;
  Tensor out = empty_like_shape(out1, out1.sizes(), at::kFloat), lse = empty_like_shape(lse1, lse1.sizes(), at::kFloat);
  if (!combine_into(out1, lse1, out2, lse2, out, lse, base)) return std::nullopt;
  return Two{out, lse};
}

bool cast_f32_bf16_into(const Tensor& src, const Tensor& dst) {
  if (!src.is_cuda() || dst.device() != src.device() || src.scalar_type() != at::kFloat || dst.scalar_type() != at::kBFloat16 ||
      src.numel() != dst.numel() || !src.is_contiguous() || !dst.is_contiguous())
    return false;
  return accepted(pith_cast_f32_bf16(src.data_ptr<float>(), dst.data_ptr(), src.numel(), stream_of(src)));
}

// ---------------------------------------------------------------------------------------------
// Per-head RMSNorm + rotary embedding

// Fields that forward and backward share; x and out contiguous.
bool norm_rope_args(pith_norm_rope_args& a, const Tensor& x, const OptTensor& weight, const Tensor& cos, const Tensor& sin, const Tensor& out, double eps) {
  if (!is_gpu_bf16(x, 4) || !x.is_contiguous()) return false;
  a.B = x.size(0); a.S = x.size(1); a.H = x.size(2); a.D = x.size(3);
  if (!cos.is_cuda() || !sin.is_cuda() || cos.device() != x.device() || sin.device() != x.device() || cos.scalar_type() != at::kBFloat16 ||
      sin.scalar_type() != at::kBFloat16 || cos.sizes() != sin.sizes() || !cos.is_contiguous() || !sin.is_contiguous())
    return false;
  if (cos.dim() == 2) {
    if (!has_shape(cos, {a.S, a.D})) return false;
    a.cs_bs = 0;
  } else {
    if (cos.dim() != 3 || (cos.size(0) != 1 && cos.size(0) != a.B) || cos.size(1) != a.S || cos.size(2) != a.D) return false;
    a.cs_bs = cos.size(0) > 1 ? a.S * a.D : 0;
  }
  if (weight) {
    if (!weight->is_cuda() || weight->device() != x.device() || !has_shape(*weight, {a.D}) || !weight->is_contiguous() ||
        !dtype_code(*weight, &a.weight_dtype))
      return false;
    a.weight = weight->data_ptr();
  }
  a.x = x.data_ptr(); a.cos = cos.data_ptr(); a.sin = sin.data_ptr(); a.out = out.data_ptr();
  a.x_bs = a.out_bs = a.S * a.H * a.D;
  a.eps = (float)eps;
  return true;
}

// dout and, with a weight, dweight (in the weight's dtype: the kernel that adds the partial sums rounds it) and the scratch.
bool norm_rope_bwd_args(pith_norm_rope_args& a, const Tensor& x, const OptTensor& weight, const Tensor& dout, const Tensor& dweight, Tensor& workspace) {
  if (!is_gpu_bf16(dout, 4) || dout.device() != x.device() || dout.sizes() != x.sizes() || !dout.is_contiguous()) return false;
  a.dout = dout.data_ptr();
  a.dout_bs = a.S * a.H * a.D;
  if (!weight) return true;
  a.dweight = dweight.data_ptr();
  a.dweight_bf16 = weight->scalar_type() == at::kBFloat16;
  a.workspace_bytes = pith_norm_rope_bwd_workspace_bytes(&a);
  workspace = empty_like_shape(x, {a.workspace_bytes}, at::kByte);
  a.workspace = workspace.data_ptr();
  return true;
}

Tensor dweight_for(const Tensor& x, const OptTensor& weight) {
  if (weight) return at::empty_like(*weight);
  return empty_like_shape(x, {0}, at::kFloat);  // placeholder: an op cannot return None
}

Tensor norm_rope_fwd(const Tensor& x, const OptTensor& weight, const Tensor& cos, const Tensor& sin, double eps) {
  if (x.is_cuda()) {
    Tensor out = at::empty_like(x, at::MemoryFormat::Contiguous);
    pith_norm_rope_args a = {};
    if (norm_rope_args(a, x, weight, cos, sin, out, eps) && accepted(pith_norm_rope_fwd(&a, stream_of(x)))) return out;
  }
  return python_body<Tensor>("norm_rope_fwd", x, weight, cos, sin, eps);
}

Two norm_rope_bwd(const Tensor& x, const OptTensor& weight, const Tensor& cos, const Tensor& sin, const Tensor& dout, double eps) {
  if (x.is_cuda()) {
    Tensor dx = at::empty_like(x, at::MemoryFormat::Contiguous), dw = dweight_for(x, weight), ws;
    pith_norm_rope_args a = {};
    if (norm_rope_args(a, x, weight, cos, sin, dx, eps) && norm_rope_bwd_args(a, x, weight, dout, dw, ws) &&
        accepted(pith_norm_rope_bwd(&a, stream_of(x))))
      return {dx, dw};
  }
  return python_body<Two>("norm_rope_bwd", x, weight, cos, sin, dout, eps);
}

Two qk_norm_rope_fwd(const Tensor& q, const Tensor& k, const OptTensor& qw, const OptTensor& kw, const Tensor& cos, const Tensor& sin, double eps) {
  if (q.is_cuda() && k.is_cuda()) {
    Tensor qo = at::empty_like(q, at::MemoryFormat::Contiguous), ko = at::empty_like(k, at::MemoryFormat::Contiguous);
    pith_norm_rope_args a = {}, b = {};
    if (k.device() == q.device() && norm_rope_args(a, q, qw, cos, sin, qo, eps) && norm_rope_args(b, k, kw, cos, sin, ko, eps) &&
        accepted(pith_norm_rope_fwd_pair(&a, &b, stream_of(q))))
      return {qo, ko};
  }
  return python_body<Two>("qk_norm_rope_fwd", q, k, qw, kw, cos, sin, eps);
}

Four qk_norm_rope_bwd(const Tensor& q, const Tensor& k, const OptTensor& qw, const OptTensor& kw, const Tensor& cos, const Tensor& sin, const Tensor& dqo,
                      const Tensor& dko, double eps) {
  if (q.is_cuda() && k.is_cuda()) {
    Tensor dq = at::empty_like(q, at::MemoryFormat::Contiguous), dk = at::empty_like(k, at::MemoryFormat::Contiguous);
    Tensor dwq = dweight_for(q, qw), dwk = dweight_for(k, kw), ws_q, ws_k;
    pith_norm_rope_args a = {}, b = {};
    if (k.device() == q.device() && norm_rope_args(a, q, qw, cos, sin, dq, eps) && norm_rope_args(b, k, kw, cos, sin, dk, eps) &&
        norm_rope_bwd_args(a, q, qw, dqo, dwq, ws_q) && norm_rope_bwd_args(b, k, kw, dko, dwk, ws_k) &&
        accepted(pith_norm_rope_bwd_pair(&a, &b, stream_of(q))))
      return {dq, dk, dwq, dwk};
  }
  return python_body<Four>("qk_norm_rope_bwd", q, k, qw, kw, cos, sin, dqo, dko, eps);
}

// ---------------------------------------------------------------------------------------------
// MLA rotary embedding + query / key / value assembly

bool assemble_tables(pith_mla_assemble_args& a, const Tensor& ref, const Tensor& cos, const Tensor& sin, const OptTensor& pos) {
  for (const Tensor* t : {&cos, &sin})
    if (!is_gpu_bf16(*t, 2) || t->device() != ref.device() || !t->is_contiguous() || t->size(1) != a.Dr) return false;
  if (cos.sizes() != sin.sizes()) return false;
  a.P = cos.size(0);
  a.cos = cos.data_ptr(); a.sin = sin.data_ptr();
  if (!pos) return a.P >= a.S;
  if (std::getenv("PITHTRAIN_AMD_CHECK_POSITIONS") != nullptr) return false;  // the Python body reads the positions back
  if (!pos->is_cuda() || pos->device() != ref.device() || pos->scalar_type() != at::kLong || pos->dim() != 2 ||
      (pos->size(0) != 1 && pos->size(0) != a.B) || pos->size(1) != a.S || (a.S > 1 && pos->stride(1) != 1))
    return false;
  a.position_ids = pos->data_ptr<int64_t>();
  a.pos_bs = pos->size(0) > 1 ? pos->stride(0) : 0;
  return true;
}

Three mla_assemble_fwd(const Tensor& q, const Tensor& kv, const Tensor& k_pe, const Tensor& cos, const Tensor& sin, const OptTensor& pos) {
  const bool shapes = is_gpu_bf16(q, 4) && is_gpu_bf16(kv, 4) && (is_gpu_bf16(k_pe, 3) || (is_gpu_bf16(k_pe, 4) && k_pe.size(2) == 1)) &&
                      kv.device() == q.device() && k_pe.device() == q.device();
  if (shapes && q.is_contiguous() && kv.is_contiguous() && k_pe.stride(-1) == 1) {
    pith_mla_assemble_args a = {};
    a.B = q.size(0); a.S = q.size(1); a.H = q.size(2); a.Dr = k_pe.size(-1);
    a.Dn = q.size(3) - a.Dr;
    a.Dv = kv.size(3) - a.Dn;
    if (a.Dn > 0 && a.Dv > 0 && kv.size(0) == a.B && kv.size(1) == a.S && kv.size(2) == a.H && k_pe.size(0) == a.B && k_pe.size(1) == a.S &&
        assemble_tables(a, q, cos, sin, pos)) {
      Tensor qo = at::empty_like(q), ko = at::empty_like(q), vo = at::empty({a.B, a.S, a.H, a.Dv}, q.options());
      a.q = q.data_ptr(); a.kv = kv.data_ptr(); a.k_pe = k_pe.data_ptr();
      a.q_out = qo.data_ptr(); a.k_out = ko.data_ptr(); a.v_out = vo.data_ptr();
      a.q_bs = a.S * a.H * (a.Dn + a.Dr);
      a.kv_bs = a.S * a.H * (a.Dn + a.Dv);
      a.k_pe_rs = a.S > 1 ? k_pe.stride(1) : a.Dr;
      a.k_pe_bs = a.B > 1 ? k_pe.stride(0) : a.S * k_pe.stride(1);
      if (accepted(pith_mla_assemble_fwd(&a, stream_of(q)))) return {qo, ko, vo};
    }
  }
  return python_body<Three>("mla_assemble_fwd", q, kv, k_pe, cos, sin, pos);
}

Three mla_assemble_bwd(const Tensor& dqo, const Tensor& dko, const Tensor& dvo, const Tensor& cos, const Tensor& sin, const OptTensor& pos, int64_t k_pe_heads) {
  const bool shapes = is_gpu_bf16(dqo, 4) && is_gpu_bf16(dko, 4) && is_gpu_bf16(dvo, 4) && dko.device() == dqo.device() && dvo.device() == dqo.device() &&
                      cos.dim() == 2;
  if (shapes && dqo.is_contiguous() && dko.is_contiguous() && dvo.is_contiguous() && dko.sizes() == dqo.sizes()) {
    pith_mla_assemble_args a = {};
    a.B = dqo.size(0); a.S = dqo.size(1); a.H = dqo.size(2); a.Dr = cos.size(1); a.Dv = dvo.size(3);
    a.Dn = dqo.size(3) - a.Dr;
    if (a.Dn > 0 && dvo.size(0) == a.B && dvo.size(1) == a.S && dvo.size(2) == a.H && assemble_tables(a, dqo, cos, sin, pos)) {
      Tensor dq = at::empty_like(dqo), dkv = at::empty({a.B, a.S, a.H, a.Dn + a.Dv}, dqo.options());
      Tensor dpe = k_pe_heads ? at::empty({a.B, a.S, 1, a.Dr}, dqo.options()) : at::empty({a.B, a.S, a.Dr}, dqo.options());
      a.dq_out = dqo.data_ptr(); a.dk_out = dko.data_ptr(); a.dv_out = dvo.data_ptr();
      a.q_out = dq.data_ptr(); a.k_out = dkv.data_ptr(); a.v_out = dpe.data_ptr();
      if (accepted(pith_mla_assemble_bwd(&a, stream_of(dqo)))) return {dq, dkv, dpe};
    }
  }
  return python_body<Three>("mla_assemble_bwd", dqo, dko, dvo, cos, sin, pos, k_pe_heads);
}

// ---------------------------------------------------------------------------------------------
// Autograd. Each formula calls the ops through the dispatcher, below autograd, so that fake tensors, functionalisation and
// torch.compile see ordinary ops. A result carries a node whenever any floating-point input requires grad, the rotary tables
// too: they receive no gradient, but a program whose tables alone require grad may still call backward().

template <typename Sig>
auto op_handle(const char* name) { return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<Sig>(); }

bool any_requires_grad(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}

Tensor or_undefined(const OptTensor& t) { return t ? *t : Tensor(); }
OptTensor or_none(const Tensor& t) { return t.defined() ? OptTensor(t) : OptTensor(); }

Two call_attn_fwd(const Tensor& q, const Tensor& k, const Tensor& v, double scale, bool causal) {
  static const auto op = op_handle<decltype(attn_fwd)>("pithtrain_amd::attn_fwd");
  return op.call(q, k, v, scale, causal);
}
struct AttnFunction : torch::autograd::Function<AttnFunction> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, double scale, bool causal) {
    at::AutoDispatchBelowADInplaceOrView guard;
    auto [o, lse] = call_attn_fwd(q, k, v, scale, causal);
    ctx->save_for_backward({q, k, v, o, lse});
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["causal"] = causal;
    ctx->mark_non_differentiable({lse});
    ctx->set_materialize_grads(false);
    return {o, lse};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    static const auto op = op_handle<decltype(attn_bwd)>("pithtrain_amd::attn_bwd");
    if (!grads[0].defined()) return {Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    const auto s = ctx->get_saved_variables();
    auto [dq, dk, dv] = op.call(s[0], s[1], s[2], s[3], s[4], grads[0], ctx->saved_data["scale"].toDouble(), ctx->saved_data["causal"].toBool());
    return {dq, dk, dv, Tensor(), Tensor()};
  }
};
Two attn_fwd_autograd(const Tensor& q, const Tensor& k, const Tensor& v, double scale, bool causal) {
  if (!any_requires_grad({&q, &k, &v})) {
    at::AutoDispatchBelowADInplaceOrView guard;
    return call_attn_fwd(q, k, v, scale, causal);
  }
  auto r = AttnFunction::apply(q, k, v, scale, causal);
  return {r[0], r[1]};
}

Tensor call_norm_rope_fwd(const Tensor& x, const OptTensor& w, const Tensor& cos, const Tensor& sin, double eps) {
  static const auto op = op_handle<decltype(norm_rope_fwd)>("pithtrain_amd::norm_rope_fwd");
  return op.call(x, w, cos, sin, eps);
}
struct NormRopeFunction : torch::autograd::Function<NormRopeFunction> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const OptTensor& w, const Tensor& cos, const Tensor& sin, double eps) {
    at::AutoDispatchBelowADInplaceOrView guard;
    ctx->save_for_backward({x, or_undefined(w), cos, sin});
    ctx->saved_data["eps"] = eps;
    return call_norm_rope_fwd(x, w, cos, sin, eps);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    static const auto op = op_handle<decltype(norm_rope_bwd)>("pithtrain_amd::norm_rope_bwd");
    const auto s = ctx->get_saved_variables();
    auto [dx, dw] = op.call(s[0], or_none(s[1]), s[2], s[3], grads[0], ctx->saved_data["eps"].toDouble());
    return {dx, s[1].defined() ? dw : Tensor(), Tensor(), Tensor(), Tensor()};
  }
};
Tensor norm_rope_fwd_autograd(const Tensor& x, const OptTensor& w, const Tensor& cos, const Tensor& sin, double eps) {
  const Tensor ww = or_undefined(w);
  if (any_requires_grad({&x, &ww, &cos, &sin})) return NormRopeFunction::apply(x, w, cos, sin, eps);
  at::AutoDispatchBelowADInplaceOrView guard;
  return call_norm_rope_fwd(x, w, cos, sin, eps);
}

Two call_qk_norm_rope_fwd(const Tensor& q, const Tensor& k, const OptTensor& qw, const OptTensor& kw, const Tensor& cos, const Tensor& sin, double eps) {
  static const auto op = op_handle<decltype(qk_norm_rope_fwd)>("pithtrain_amd::qk_norm_rope_fwd");
  return op.call(q, k, qw, kw, cos, sin, eps);
}
struct QkNormRopeFunction : torch::autograd::Function<QkNormRopeFunction> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const OptTensor& qw, const OptTensor& kw, const Tensor& cos,
                               const Tensor& sin, double eps) {
    at::AutoDispatchBelowADInplaceOrView guard;
    ctx->save_for_backward({q, k, or_undefined(qw), or_undefined(kw), cos, sin});
    ctx->saved_data["eps"] = eps;
    auto [qo, ko] = call_qk_norm_rope_fwd(q, k, qw, kw, cos, sin, eps);
    return {qo, ko};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    static const auto op = op_handle<decltype(qk_norm_rope_bwd)>("pithtrain_amd::qk_norm_rope_bwd");
    const auto s = ctx->get_saved_variables();
    auto [dq, dk, dwq, dwk] = op.call(s[0], s[1], or_none(s[2]), or_none(s[3]), s[4], s[5], grads[0], grads[1], ctx->saved_data["eps"].toDouble());
    return {dq, dk, s[2].defined() ? dwq : Tensor(), s[3].defined() ? dwk : Tensor(), Tensor(), Tensor(), Tensor()};
  }
};
Two qk_norm_rope_fwd_autograd(const Tensor& q, const Tensor& k, const OptTensor& qw, const OptTensor& kw, const Tensor& cos, const Tensor& sin, double eps) {
  const Tensor a = or_undefined(qw), b = or_undefined(kw);
  if (any_requires_grad({&q, &k, &a, &b, &cos, &sin})) {
    auto r = QkNormRopeFunction::apply(q, k, qw, kw, cos, sin, eps);
    return {r[0], r[1]};
  }
  at::AutoDispatchBelowADInplaceOrView guard;
  return call_qk_norm_rope_fwd(q, k, qw, kw, cos, sin, eps);
}

Three call_mla_assemble_fwd(const Tensor& q, const Tensor& kv, const Tensor& k_pe, const Tensor& cos, const Tensor& sin, const OptTensor& pos) {
  static const auto op = op_handle<decltype(mla_assemble_fwd)>("pithtrain_amd::mla_assemble_fwd");
  return op.call(q, kv, k_pe, cos, sin, pos);
}
struct MlaAssembleFunction : torch::autograd::Function<MlaAssembleFunction> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& kv, const Tensor& k_pe, const Tensor& cos, const Tensor& sin,
                               const OptTensor& pos) {
    at::AutoDispatchBelowADInplaceOrView guard;
    ctx->save_for_backward({cos, sin, or_undefined(pos)});
    ctx->saved_data["k_pe_heads"] = (int64_t)(k_pe.dim() == 4 ? 1 : 0);
    auto [qo, ko, vo] = call_mla_assemble_fwd(q, kv, k_pe, cos, sin, pos);
    return {qo, ko, vo};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    static const auto op = op_handle<decltype(mla_assemble_bwd)>("pithtrain_amd::mla_assemble_bwd");
    const auto s = ctx->get_saved_variables();
    auto [dq, dkv, dpe] = op.call(grads[0], grads[1], grads[2], s[0], s[1], or_none(s[2]), ctx->saved_data["k_pe_heads"].toInt());
    return {dq, dkv, dpe, Tensor(), Tensor(), Tensor()};
  }
};
Three mla_assemble_fwd_autograd(const Tensor& q, const Tensor& kv, const Tensor& k_pe, const Tensor& cos, const Tensor& sin, const OptTensor& pos) {
  if (any_requires_grad({&q, &kv, &k_pe, &cos, &sin})) {
    auto r = MlaAssembleFunction::apply(q, kv, k_pe, cos, sin, pos);
    return {r[0], r[1], r[2]};
  }
  at::AutoDispatchBelowADInplaceOrView guard;
  return call_mla_assemble_fwd(q, kv, k_pe, cos, sin, pos);
}

// One rank's ring share as one node. What its Python counterpart (RingAttentionLocalFunc) spends on a dozen chunk tensors
// outlasts the kernels of a short share: forward + backward of 64 rows, 16 heads of 192 in two parts, rank 2 of 4 177 -> 138 us (of
// which 108 are the engine handing out ten gradients); 1021 rows 165 -> 157 us, now the length of its kernels.
// Inputs: q, then the visited chunks of K, of V and, if keys come in two parts, of k_pe.
using OptTensors = std::vector<OptTensor>;

int64_t visited_chunks(int64_t rank, int64_t cp, bool zigzag) { return zigzag ? cp : rank + 1; }  // the first ones, by rank

struct RingFunction : torch::autograd::Function<RingFunction> {
  // chunk lists of cp entries from the flat inputs, whose first chunk is at `first`
  static std::vector<OptTensors> chunk_lists(at::TensorList in, size_t first, int64_t cp, int64_t visited) {
    std::vector<OptTensors> lists((in.size() - first) / visited, OptTensors(cp));
    for (size_t kind = 0; kind < lists.size(); ++kind)
      for (int64_t j = 0; j < visited; ++j) lists[kind][j] = in[first + kind * visited + j];
    return lists;
  }
  static std::optional<OptTensors> part_two(const std::vector<OptTensors>& lists) {
    return lists.size() == 3 ? std::optional<OptTensors>(lists[2]) : std::nullopt;
  }
  static Tensor forward(AutogradContext* ctx, at::TensorList in, double scale, int64_t rank, int64_t cp, bool zigzag) {
    at::AutoDispatchBelowADInplaceOrView guard;
    const auto lists = chunk_lists(in, 1, cp, visited_chunks(rank, cp, zigzag));
    auto done = ring_forward(in[0], lists[0], lists[1], part_two(lists), scale, rank, cp, zigzag);
    if (!done) done = python_body<Two>("ring_forward_local", in[0], lists[0], lists[1], scale, rank, cp, zigzag, part_two(lists));
    variable_list saved = {std::get<0>(*done), std::get<1>(*done)};
    saved.insert(saved.end(), in.begin(), in.end());
    ctx->save_for_backward(std::move(saved));
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["rank"] = rank;
    ctx->saved_data["cp"] = cp;
    ctx->saved_data["zigzag"] = zigzag;
    return std::get<0>(*done);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    at::AutoDispatchBelowADInplaceOrView guard;
    const auto s = ctx->get_saved_variables();  // out, lse, q, chunks
    const double scale = ctx->saved_data["scale"].toDouble();
    const int64_t rank = ctx->saved_data["rank"].toInt(), cp = ctx->saved_data["cp"].toInt();
    const bool zigzag = ctx->saved_data["zigzag"].toBool();
    const int64_t visited = visited_chunks(rank, cp, zigzag);
    const Tensor &out = s[0], &lse = s[1], &q = s[2];
    const auto lists = chunk_lists(s, 3, cp, visited);
    std::optional<RingGrads> g;
    // Whether a share or its steps hand dS over is the Python body's decision where they could.
    const bool whole_keys = q.size(3) == 128 || (q.size(3) == 192 && !part_two(lists));
    if (share_ds_bytes(q, lists[0], lists[1], part_two(lists), rank, cp, zigzag) == 0 &&
        (!whole_keys || (q.size(3) == 192 && !step_of_192_hands_over(q.size(0), q.size(1), q.size(2), lists[0][0]->size(2), rank, cp, zigzag, compute_units(q.device().index())))))
      g = ring_backward(grads[0], q, out, lse, lists[0], lists[1], part_two(lists), scale, rank, cp, zigzag, {});
    if (!g) g = python_body<RingGrads>("ring_backward_local", grads[0], q, out, lse, lists[0], lists[1], scale, rank, cp, zigzag, part_two(lists));
    variable_list r = {std::get<0>(*g)};
    for (const OptTensors* kind : {&std::get<1>(*g), &std::get<2>(*g), &std::get<3>(*g)})
      for (int64_t j = 0; j < visited && j < (int64_t)kind->size(); ++j) r.push_back(or_undefined((*kind)[j]));
    r.resize(s.size() - 2 + 4);  // scale, rank, cp, zigzag
    return r;
  }
};

// None where the Python function has to do: CPU tensors and missing chunks (it words the errors), and tensors or modes that
// look at every operation (fake, batched and functional tensors, dispatch modes, tracing, forward-mode gradients).
OptTensor ring_attention(const Tensor& q, const OptTensors& ks, const OptTensors& vs, const std::optional<OptTensors>& pes, double scale, int64_t rank,
                         int64_t cp, bool zigzag) {
  if (!(c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set).empty()) return {};
  if (rank < 0 || rank >= cp || (int64_t)ks.size() != cp || (int64_t)vs.size() != cp || (pes && (int64_t)pes->size() != cp)) return {};
  constexpr c10::DispatchKeySet watching({c10::DispatchKey::Python, c10::DispatchKey::Functionalize, c10::DispatchKey::FuncTorchBatched,
                                          c10::DispatchKey::BatchedNestedTensor, c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Batched});
  const auto plain = [&](const OptTensor& t) { return t && t->is_cuda() && !t->key_set().has_any(watching) && !t->_fw_grad(0).defined(); };
  if (!plain(q) || q.dim() != 4) return {};
  variable_list in = {q};
  bool recorded = q.requires_grad();
  for (const OptTensors* kind : {&ks, &vs, pes ? &*pes : nullptr})
    for (int64_t j = 0; kind && j < visited_chunks(rank, cp, zigzag); ++j) {
      if (!plain((*kind)[j])) return {};
      in.push_back(*(*kind)[j]);
      recorded |= in.back().requires_grad();
    }
  if (recorded && at::GradMode::is_enabled()) return RingFunction::apply(at::TensorList(in), scale, rank, cp, zigzag);
  at::AutoDispatchBelowADInplaceOrView guard;
  if (auto done = ring_forward(q, ks, vs, pes, scale, rank, cp, zigzag)) return std::get<0>(*done);
  return std::get<0>(python_body<Two>("ring_forward_local", q, ks, vs, scale, rank, cp, zigzag, pes));
}

// The backward ops have no derivative of their own: under create_graph their results carry a node that raises when somebody
// differentiates through it (without one the dispatcher would only warn and leave the second-order part out).
struct NoSecondDerivative : torch::autograd::Function<NoSecondDerivative> {
  static variable_list forward(AutogradContext*, at::TensorList, const std::function<variable_list()>& call) { return call(); }
  static variable_list backward(AutogradContext*, variable_list) {
    TORCH_CHECK(false, "Trying to backward through the backward of a pithtrain_amd operator: second derivatives are not implemented");
  }
};

void collect(variable_list& l, const Tensor& t) {
  if (t.defined()) l.push_back(t);
}
void collect(variable_list& l, const OptTensor& t) { collect(l, or_undefined(t)); }
template <typename T>
std::enable_if_t<std::is_arithmetic_v<T>> collect(variable_list&, T) {}

template <typename... Tensors>
std::tuple<Tensors...> as_tuple(const variable_list& l) {
  size_t i = 0;
  return std::tuple<Tensors...>{(Tensors)l[i++]...};
}

template <auto BODY>
struct BackwardOp;
template <typename... Tensors, typename... Args, std::tuple<Tensors...> (*BODY)(Args...)>
struct BackwardOp<BODY> {
  template <const char* NAME>
  static std::tuple<Tensors...> call(Args... args) {
    static const auto op = op_handle<std::tuple<Tensors...>(Args...)>(NAME);
    bool recorded = false;
    variable_list inputs;
    if (at::GradMode::is_enabled()) {
      (collect(inputs, args), ...);
      for (const Tensor& t : inputs) recorded |= t.requires_grad();
    }
    const auto below = [&] {
      at::AutoDispatchBelowADInplaceOrView guard;
      return op.call(args...);
    };
    if (!recorded) return below();
    return as_tuple<Tensors...>(NoSecondDerivative::apply(at::TensorList(inputs), std::function<variable_list()>([&] {
      return std::apply([](const auto&... t) { return variable_list{t...}; }, below());
    })));
  }
};

constexpr char kAttnBwd[] = "pithtrain_amd::attn_bwd", kNormRopeBwd[] = "pithtrain_amd::norm_rope_bwd",
               kQkNormRopeBwd[] = "pithtrain_amd::qk_norm_rope_bwd", kMlaAssembleBwd[] = "pithtrain_amd::mla_assemble_bwd";

}  // namespace

TORCH_LIBRARY(pithtrain_amd, m) {
  m.def("attn_fwd(Tensor q, Tensor k, Tensor v, float softmax_scale, bool causal) -> (Tensor, Tensor)");
  m.def("attn_bwd(Tensor q, Tensor k, Tensor v, Tensor o, Tensor lse, Tensor dout, float softmax_scale, bool causal) -> (Tensor, Tensor, Tensor)");
  m.def("norm_rope_fwd(Tensor x, Tensor? weight, Tensor cos, Tensor sin, float eps) -> Tensor");
  m.def("norm_rope_bwd(Tensor x, Tensor? weight, Tensor cos, Tensor sin, Tensor dout, float eps) -> (Tensor, Tensor)");
  m.def("qk_norm_rope_fwd(Tensor q, Tensor k, Tensor? q_weight, Tensor? k_weight, Tensor cos, Tensor sin, float eps) -> (Tensor, Tensor)");
  m.def("qk_norm_rope_bwd(Tensor q, Tensor k, Tensor? q_weight, Tensor? k_weight, Tensor cos, Tensor sin, Tensor dq_out, Tensor dk_out, float eps) "
        "-> (Tensor, Tensor, Tensor, Tensor)");
  m.def("mla_assemble_fwd(Tensor q, Tensor kv, Tensor k_pe, Tensor cos, Tensor sin, Tensor? position_ids) -> (Tensor, Tensor, Tensor)");
  m.def("mla_assemble_bwd(Tensor dq_out, Tensor dk_out, Tensor dv_out, Tensor cos, Tensor sin, Tensor? position_ids, int k_pe_heads) "
        "-> (Tensor, Tensor, Tensor)");
}

// CPU tensors are refused by the Python bodies (there is no CPU path); they reach them through the same functions.
#define PITH_IMPL(key)                               \
  TORCH_LIBRARY_IMPL(pithtrain_amd, key, m) {        \
    m.impl("attn_fwd", &attn_fwd);                   \
    m.impl("attn_bwd", &attn_bwd);                   \
    m.impl("norm_rope_fwd", &norm_rope_fwd);         \
    m.impl("norm_rope_bwd", &norm_rope_bwd);         \
    m.impl("qk_norm_rope_fwd", &qk_norm_rope_fwd);   \
    m.impl("qk_norm_rope_bwd", &qk_norm_rope_bwd);   \
    m.impl("mla_assemble_fwd", &mla_assemble_fwd);   \
    m.impl("mla_assemble_bwd", &mla_assemble_bwd);   \
  }
PITH_IMPL(CUDA)
PITH_IMPL(CPU)
#undef PITH_IMPL

TORCH_LIBRARY_IMPL(pithtrain_amd, Autograd, m) {
  m.impl("attn_fwd", &attn_fwd_autograd);
  m.impl("norm_rope_fwd", &norm_rope_fwd_autograd);
  m.impl("qk_norm_rope_fwd", &qk_norm_rope_fwd_autograd);
  m.impl("mla_assemble_fwd", &mla_assemble_fwd_autograd);
  m.impl("attn_bwd", &BackwardOp<&attn_bwd>::call<kAttnBwd>);
  m.impl("norm_rope_bwd", &BackwardOp<&norm_rope_bwd>::call<kNormRopeBwd>);
  m.impl("qk_norm_rope_bwd", &BackwardOp<&qk_norm_rope_bwd>::call<kQkNormRopeBwd>);
  m.impl("mla_assemble_bwd", &BackwardOp<&mla_assemble_bwd>::call<kMlaAssembleBwd>);
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  TORCH_CHECK(pith_version() == PITH_VERSION, "_pith_torch.so was built for interface version ", PITH_VERSION, " of libpith_hip.so, found ",
              pith_version(), ": build both again");
  m.def("set_bodies", [](py::dict d) { bodies().attr("update")(d); }, "Registers the Python bodies of ops (name -> function).");
  // These allocate and launch, either of which can block (a full queue): other Python threads run meanwhile.
  using Unlocked = py::call_guard<py::gil_scoped_release>;
  m.def("attn_fwd_into", &attn_fwd_into, Unlocked());
  m.def("attn_bwd_delta_into", &attn_bwd_delta_into, Unlocked());
  m.def("attn_bwd_dkdv_into", &attn_bwd_dkdv_into, Unlocked());
  m.def("attn_bwd_dq_into", &attn_bwd_dq_into, Unlocked());
  m.def("attn_bwd_pair_into", &attn_bwd_pair_into, Unlocked());
  m.def("ring_forward", &ring_forward, Unlocked());
  m.def("ring_backward", &ring_backward, py::arg("dout"), py::arg("q"), py::arg("out"), py::arg("lse"), py::arg("ks"), py::arg("vs"), py::arg("pes"),
        py::arg("scale"), py::arg("rank"), py::arg("cp"), py::arg("zigzag"), py::arg("ds") = py::none(), Unlocked());
  m.def("share_ds_bytes", &share_ds_bytes);
  m.def("share_of_192_pays", &share_of_192_pays);
  m.def("ring_attention", &ring_attention, Unlocked());
  m.def("combine_into", &combine_into, Unlocked());
  m.def("combine_new", &combine_new, Unlocked());
  m.def("cast_f32_bf16_into", &cast_f32_bf16_into, Unlocked());
  m.def("accepted", &accepted);
  m.def("share_forward_in_one", &share_forward_in_one);
  m.def("share_backward_in_one", &share_backward_in_one);
  m.def("ds_handover_pays", &ds_handover_pays);
  m.def("ds_handover_pays_192", &ds_handover_pays_192);
  m.def("step_of_192_hands_over", &step_of_192_hands_over);
  m.def("share_hands_over", &share_hands_over, py::arg("b"), py::arg("rows"), py::arg("hq"), py::arg("hkv"), py::arg("steps"), py::arg("cus"),
        py::arg("dqk") = 128);
}
