// Entry point of the query-gradient step of one chunk attention backward for gfx950 (against an external, ring-combined
// base-2 LSE and delta = rowsum(O*dO)): argument checks shared with the dK/dV step and the choice of a kernel. Numerics of
// all kernels follow pithtrain/operators/mla/triton.py:205-266 (non-causal :392-441).
#include "attn_bwd_common.h"

namespace pith {
namespace {

// Recomputing dQ kernels: 128-row workgroups either way. Two 4-wave workgroups per compute unit (attn_bwd_dq_duo.hip), or
// one of 8 waves whose pairs split every tile's keys (attn_bwd_dq_direct.hip, "half"). Measured, microseconds:
//                                              duo    half
//   d128  1 x 4096 x 32 heads causal           176    197        d192  1 x 4096 x 128 heads causal     1105   1210
//         1 x 2048 x 32, 512 WGs, causal       65     58               1 x 4096 x 16, 512 WGs, causal  179    136
//         1 x 1024 x 32, 256 WGs, no mask      32     30               2048 x 4096 x 16, 256 WGs       139    120
//         1 x 1536 x 32, 384 WGs, no mask      56     69               4096 x 2048 x 16, 512 WGs       119    130
//         1 x 256 x 32                         12.1   12.7             1 x 256 x 16                    15.9   16.4
// So the split keys pay where a workgroup has its compute unit to itself: grids of up to one workgroup per unit, and under
// the mask, where the heavy half of the workgroups ends up alone, of up to two for long streams (the same lines as in the
// forward). 64 features always use duo (three workgroups fit a unit; no split-key kernel exists).
bool dq_split_keys(const pith_attn_bwd_args* a) {
  if (a->Dqk == 64) return false;
  const int64_t cus = compute_units_or_default();
  const int64_t wgs = ((a->Sq + 127) / 128) * a->Hq * a->B;
  return wgs <= cus ? a->Skv > 256 : a->causal && wgs <= 2 * cus && a->Skv >= 1536;
}

}  // namespace

bool ds_usable(const pith_attn_bwd_args* a) {
  // (192 features: the field was ignored before there was a hand-over, so what callers left in it is no error)
  return a->ds && ds_bytes_for(a) > 0 && a->ds_bytes >= ds_bytes_for(a) && (a->Dqk != 192 || (uintptr_t)a->ds % 256 == 0);
}

int validate_bwd(const pith_attn_bwd_args* a, const char* who, bool need_dq, bool need_dkv) {
  if (!a) return fail(PITH_ERR_NULL_POINTER, "%s: args is NULL", who);
  if (!a->q || !a->k || !a->v || !a->dout || !a->lse || !a->delta)
    return fail(PITH_ERR_NULL_POINTER, "%s: NULL input tensor pointer", who);
  if (need_dq && !a->dq) return fail(PITH_ERR_NULL_POINTER, "%s: dq is NULL", who);
  if (need_dkv && (!a->dk || !a->dv)) return fail(PITH_ERR_NULL_POINTER, "%s: dk or dv is NULL", who);
  if (a->B <= 0 || a->Sq <= 0 || a->Skv <= 0 || a->Hq <= 0 || a->Hkv <= 0)
    return fail(PITH_ERR_BAD_SHAPE, "%s: B=%lld Sq=%lld Skv=%lld Hq=%lld Hkv=%lld must all be positive", who,
                (long long)a->B, (long long)a->Sq, (long long)a->Skv, (long long)a->Hq, (long long)a->Hkv);
  if (a->Hq % a->Hkv != 0)
    return fail(PITH_ERR_BAD_SHAPE, "%s: Hq=%lld is not a multiple of Hkv=%lld", who, (long long)a->Hq, (long long)a->Hkv);
  if ((a->q_row_heads && (a->q_row_heads < a->Hq || a->q_row_heads > 65535)) ||
      (a->kv_row_heads && (a->kv_row_heads < a->Hkv || a->kv_row_heads > 65535)))
    return fail(PITH_ERR_BAD_SHAPE, "%s: q_row_heads=%lld / kv_row_heads=%lld must be 0 or at least Hq=%lld / Hkv=%lld", who,
                (long long)a->q_row_heads, (long long)a->kv_row_heads, (long long)a->Hq, (long long)a->Hkv);
  if (a->k_pe && (a->q_row_heads > a->Hq || a->kv_row_heads > a->Hkv))
    return fail(PITH_ERR_UNSUPPORTED, "%s: keys in two parts cannot be combined with a head range of wider tensors", who);
  if (a->dkv_zero_tail < 0 || a->dkv_zero_tail > (1 << 24))
    return fail(PITH_ERR_BAD_SHAPE, "%s: dkv_zero_tail=%lld out of range", who, (long long)a->dkv_zero_tail);
  if (a->causal && a->Sq != a->Skv)
    return fail(PITH_ERR_UNSUPPORTED, "%s: causal needs Sq == Skv (got %lld, %lld)", who, (long long)a->Sq, (long long)a->Skv);
  if (a->Sq > (1 << 24) || a->Skv > (1 << 24) || a->Hq > 65535 || a->B > 65535 ||
      ((a->Sq + 31) / 32) * a->Hq * a->B > 0x7fffffffLL)
    return fail(PITH_ERR_UNSUPPORTED, "%s: sequence, head or batch count beyond the launch grid limits", who);
  if (!(a->scale > 0.f) || !(a->scale < INFINITY))
    return fail(PITH_ERR_BAD_SHAPE, "%s: scale=%g must be positive and finite", who, (double)a->scale);
  const int dt = need_dq ? a->dq_dtype : a->dkv_dtype;
  if (dt != PITH_BF16 && dt != PITH_F32) return fail(PITH_ERR_BAD_DTYPE, "%s: output dtype %d is not bf16/fp32", who, dt);
  if (!aligned16(a->q) || !aligned16(a->k) || !aligned16(a->v) || !aligned16(a->dout) || a->q_bs % 8 || a->k_bs % 8 ||
      a->v_bs % 8 || a->dout_bs % 8)
    return fail(PITH_ERR_MISALIGNED, "%s: input pointers / batch strides must keep 16-byte alignment", who);
  if (need_dq && (!aligned16(a->dq) || a->dq_bs % 8))
    return fail(PITH_ERR_MISALIGNED, "%s: dq pointer / batch stride must keep 16-byte alignment", who);
  if (need_dkv && (!aligned16(a->dk) || !aligned16(a->dv) || a->dk_bs % 8 || a->dv_bs % 8))
    return fail(PITH_ERR_MISALIGNED, "%s: dk/dv pointers / batch strides must keep 16-byte alignment", who);
  if (a->k_pe) {
    if (a->Dqk != 192 || a->Dv != 128)
      return fail(PITH_ERR_UNSUPPORTED, "%s: keys in two parts (k_pe) need head dims (192, 128), got (%lld, %lld)", who,
                  (long long)a->Dqk, (long long)a->Dv);
    if (!aligned16(a->k_pe) || a->k_pe_bs % 8 || a->k_pe_rs % 8 || a->k_pe_rs < 64)
      return fail(PITH_ERR_MISALIGNED, "%s: k_pe pointer / strides must keep 16-byte alignment (row stride >= 64)", who);
  }
  const bool dims_ok = (a->Dqk == 128 && a->Dv == 128) || (a->Dqk == 192 && a->Dv == 128) || (a->Dqk == 64 && a->Dv == 64);
  if (!dims_ok)
    return fail(PITH_ERR_UNSUPPORTED, "%s: head dims (Dqk=%lld, Dv=%lld) not in {(64,64),(128,128),(192,128)}", who,
                (long long)a->Dqk, (long long)a->Dv);
  return PITH_OK;
}

BwdParams make_bwd_params(const pith_attn_bwd_args* a) {
  BwdParams p;
  p.q = (const __bf16*)a->q; p.k = (const __bf16*)a->k; p.v = (const __bf16*)a->v; p.dout = (const __bf16*)a->dout;
  p.lse = a->lse; p.delta = a->delta; p.dq = a->dq; p.dk = a->dk; p.dv = a->dv;
  p.Sq = (int)a->Sq; p.Skv = (int)a->Skv; p.Hq = (int)a->Hq; p.Hkv = (int)a->Hkv; p.group = (int)(a->Hq / a->Hkv); p.B = (int)a->B;
  p.HqT = (int)(a->q_row_heads ? a->q_row_heads : a->Hq);
  p.HkvT = (int)(a->kv_row_heads ? a->kv_row_heads : a->Hkv);
  p.tiles = p.q_tiles = 0;
  p.q_bs = a->q_bs; p.k_bs = a->k_bs; p.v_bs = a->v_bs; p.dout_bs = a->dout_bs;
  p.dq_bs = a->dq_bs; p.dk_bs = a->dk_bs; p.dv_bs = a->dv_bs; p.lse_bs = a->lse_bs; p.lse_hs = a->lse_hs;
  p.scale = a->scale;
  p.kappa = a->scale * 1.44269504088896340736f;
  p.accumulate = p.accumulate_dq = 0;
  // (fp32 results are updated by later steps)
  p.through_dkv = a->dkv_dtype == PITH_BF16 && through_results(a->B * a->Skv * a->Hkv * (a->Dqk + a->Dv) * 2);
  p.through_dq = a->dq_dtype == PITH_BF16 && through_results(a->B * a->Sq * a->Hq * a->Dqk * 2);
  p.through_parts = 0;
  p.chunked = bwd_chunked_tiles(a->causal != 0, a->Hq != a->Hkv, ds_usable(a));
  p.split = 1;
  p.ws_dk = nullptr;
  p.ws_dv = nullptr;
  p.k_pe = (const __bf16*)a->k_pe; p.k_pe_bs = a->k_pe_bs; p.k_pe_rs = a->k_pe_rs;
  p.ws_dkpe = nullptr;
  p.ds = nullptr;
  p.ds_qt = (int)((a->Sq + 63) / 64);
  p.ds_kb = (int)((a->Skv + kDkdvBlockN - 1) / kDkdvBlockN);
  p.ds_hs = (a->causal ? ds_tile_start<true>(p.ds_qt, p.ds_kb) : ds_tile_start<false>(p.ds_qt, p.ds_kb)) * kDsBlockBytes;
  p.dq_final = nullptr; p.dq_final_bs = 0; p.final_r0 = p.final_r1 = 0;
  p.zero_tail = 0; p.main_blocks = 0x7fffffff; p.dk_pe = nullptr; p.dk_pe_bs = 0; p.walk_desc = 0;
  return p;
}

int64_t ds_bytes_for(const pith_attn_bwd_args* a) {
  if (!a || (a->Dqk != 128 && a->Dqk != 192) || a->Dv != 128 || a->k_pe || a->B <= 0 || a->Hq <= 0 || a->Sq <= 0 || a->Skv <= 0) return 0;
  if (a->Dqk == 192 && a->Sq <= dq_ds_rows(192) / 2) return 0;  // half of every dQ workgroup would be empty
  const int qt = (int)((a->Sq + 63) / 64), kb = (int)((a->Skv + kDkdvBlockN - 1) / kDkdvBlockN);
  // a causal call (Sq == Skv) keeps only the key blocks at or below the diagonal of every query tile
  const int64_t blocks = a->causal ? ds_tile_start<true>(qt, kb) : ds_tile_start<false>(qt, kb);
  return a->B * a->Hq * blocks * kDsBlockBytes;
}

}  // namespace pith

using namespace pith;

extern "C" int64_t pith_attn_bwd_ds_bytes(const pith_attn_bwd_args* a) { return ds_bytes_for(a); }

namespace pith {

// What the dQ call adds to the shared parameters: its accumulation and the rows it finishes.
int prepare_dq(const pith_attn_bwd_args* a, BwdParams* p, const char* who) {
  p->accumulate_dq = a->accumulate_dq;
  if (!a->dq_final) return PITH_OK;
  if (a->dq_dtype != PITH_F32 || a->Dv != 128 || (a->Dqk != 128 && a->Dqk != 192))
    return fail(PITH_ERR_UNSUPPORTED, "%s: dq_final needs an fp32 dq and head dims (128,128) or (192,128)", who);
  if (!aligned16(a->dq_final) || a->dq_final_bs % 8)
    return fail(PITH_ERR_MISALIGNED, "%s: dq_final pointer / batch stride must keep 16-byte alignment", who);
  int64_t r0 = a->dq_final_rows[0], r1 = a->dq_final_rows[1];
  if (r0 == 0 && r1 == 0) r1 = a->Sq;
  if (r0 < 0 || r1 < r0 || r1 > a->Sq || r0 % 32 || (r1 % 32 && r1 != a->Sq))
    return fail(PITH_ERR_BAD_SHAPE, "%s: dq_final_rows = [%lld, %lld) must lie within the %lld query rows on multiples of 32", who,
                (long long)a->dq_final_rows[0], (long long)a->dq_final_rows[1], (long long)a->Sq);
  p->dq_final = reinterpret_cast<__bf16*>(a->dq_final);
  p->dq_final_bs = a->dq_final_bs;
  p->final_r0 = (int)r0;
  p->final_r1 = (int)r1;
  return PITH_OK;
}

}  // namespace pith

extern "C" int pith_attn_bwd_dq(const pith_attn_bwd_args* a, pith_stream_t stream) {
  const char* who = "pith_attn_bwd_dq";
  if (const int rc = validate_bwd(a, who, true, false)) return rc;
  BwdParams p = make_bwd_params(a);
  if (const int rc = prepare_dq(a, &p, who)) return rc;
  hipStream_t st = (hipStream_t)stream;
  const bool f32 = a->dq_dtype == PITH_F32;
  begin_launch();
  if (ds_usable(a)) {
    // dS was left by the dK/dV call of the same chunk: one product instead of three
    if ((uintptr_t)a->ds % 256) return fail(PITH_ERR_MISALIGNED, "%s: ds must be 256-byte aligned", who);
    p.ds = reinterpret_cast<char*>(a->ds);
    const int rows = dq_ds_rows((int)a->Dqk);
    p.q_tiles = (int)((a->Sq + rows - 1) / rows);
    launch_dq_from_ds(p, (int)a->Dqk, a->causal != 0, f32, st);
  } else if (dq_split_keys(a)) {
    launch_dq_direct(p, (int)a->Dqk, a->causal != 0, f32, st);
  } else {
    launch_dq_duo(p, (int)a->Dqk, a->causal != 0, f32, st);
  }
  return check_launch(who);
}
