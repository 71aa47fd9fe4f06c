// The per-token operators of the `xenc` namespace, defined and implemented in C++ so that a
// decode call costs one dispatcher hop into the C ABI (include/xenc_hip.h): no Python in the
// call, outputs allocated by torch's caching allocator, torch's current HIP stream of the query's
// device.  Their fake (meta) kernels are registered from Python (kv_skill_v2_amd/torch_ops.py),
// as are the prefill operators.  Host code only: built with the system C++ compiler against
// torch's headers into libxenc_torch.so, next to libxenc_hip.so, whose C ABI it calls.
//
//   xenc::route_topk          LibraryInjector.route (xenc/injector.py:220-229) for few rows
//   xenc::library_read        the read of LibraryInjector._branch (xenc/injector.py:236-265)
//   xenc::route_read          both in one call (the top-k inside the read kernel when it can)
//   xenc::read_entries        the read of many rows by their routed (row, chunk) pairs, no gradient
//   xenc::library_read_entries, library_read_entries_bwd   routing + that read, and its dQ: its
//                             autograd is here too (registered from Python, a call with this many
//                             arguments spent 95 us of a small training step on its schema)
//   xenc::hook_query, hook_write, hook_add   a hooked layer's query, update and residual add around
//                             the read, for steps without a gradient
//   xenc::hook_layer          a whole hooked layer of a decode step: the above and route_read
//   xenc::paged_decode_joint  DecodeReader.__call__ (xenc/d23_read_kernels.py:145-160)
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/library.h>

#include <algorithm>
#include <string>
#include <tuple>

#include "xenc_hip.h"

namespace {

// Error codes of the C ABI as Python exceptions: argument errors are ValueError, a failed
// launch RuntimeError (the same mapping as kv_skill_v2_amd._lib.check).
void check(int rc, const char* what) {
  if (rc == XENC_OK) return;
  std::string msg = std::string(what) + ": " + xenc_strerror(rc);
  if (rc == XENC_EHIP) msg += " (hipError " + std::to_string(xenc_last_hip_error()) + ")";
  if (rc == XENC_EINVAL || rc == XENC_ENULL || rc == XENC_EALIGN || rc == XENC_EWORKSPACE ||
      rc == XENC_ESCRATCH)
    TORCH_CHECK_VALUE(false, msg);
  TORCH_CHECK(false, msg);
}

void* stream_of(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

template <class T>
T* ptr(const at::Tensor& t) {
  return static_cast<T*>(t.data_ptr());
}

int as_int(const c10::SymInt& v) { return static_cast<int>(v.expect_int()); }

at::TensorOptions f32(const at::Tensor& like) { return like.options().dtype(at::kFloat); }
at::TensorOptions i32(const at::Tensor& like) { return like.options().dtype(at::kInt); }

std::tuple<at::Tensor, at::Tensor, at::Tensor> route_topk(const at::Tensor& q, const at::Tensor& S,
                                                          const at::Tensor& chunk_ptr, const at::Tensor& q_group,
                                                          c10::SymInt top_k, double route_temp, c10::SymInt cmax,
                                                          c10::SymInt kk) {
  const c10::DeviceGuard guard(q.device());
  const int64_t M = q.size(0), d = q.size(1);
  const int C = as_int(cmax), K = as_int(kk);
  at::Tensor w = at::empty({M, C}, f32(q)), idx = at::empty({M, K}, i32(q)), wsel = at::empty({M, K}, f32(q));
  if (M)
    check(xenc_route_topk(ptr<const float>(q), q.stride(0), (int)M, (int)d, ptr<const float>(S),
                          ptr<const int>(chunk_ptr), ptr<const int>(q_group), (int)chunk_ptr.numel() - 1,
                          as_int(top_k), (float)route_temp, ptr<float>(w), w.stride(0), ptr<int>(idx),
                          ptr<float>(wsel), K, stream_of(q)),
          "xenc_route_topk");
  return {w, idx, wsel};
}

at::Tensor library_read(const at::Tensor& q, const at::Tensor& pages, const at::Tensor& chunk_page,
                        const at::Tensor& chunk_nvalid, const at::Tensor& chunk_ptr, const at::Tensor& q_group,
                        const at::Tensor& idx, const at::Tensor& w_sel, double read_temp, bool softmax,
                        c10::SymInt nsplit, at::Tensor& workspace, c10::SymInt max_rows) {
  const c10::DeviceGuard guard(q.device());
  const int64_t M = q.size(0), d = pages.size(-1), K = idx.size(1);
  at::Tensor r = at::empty({M, d}, f32(q));
  if (M == 0 || K == 0) return r.zero_();
  check(xenc_library_read_decode(ptr<const float>(q), q.stride(0), (int)M, (int)d, pages.data_ptr(),
                                 (int)pages.size(1), pages.stride(0), ptr<const int>(chunk_page),
                                 ptr<const int>(chunk_nvalid), ptr<const int>(chunk_ptr), ptr<const int>(q_group),
                                 (int)chunk_ptr.numel() - 1, ptr<const int>(idx), ptr<const float>(w_sel), (int)K,
                                 (float)read_temp, softmax ? 1 : 0, as_int(nsplit), ptr<float>(r), r.stride(0),
                                 workspace.data_ptr(), (size_t)workspace.numel(), as_int(max_rows), stream_of(q)),
        "xenc_library_read_decode");
  return r;
}

std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> route_read(
    const at::Tensor& q, const at::Tensor& S, const at::Tensor& pages, const at::Tensor& chunk_page,
    const at::Tensor& chunk_nvalid, const at::Tensor& chunk_ptr, const at::Tensor& q_group, c10::SymInt top_k,
    double route_temp, c10::SymInt cmax, c10::SymInt kk, double read_temp, bool softmax, c10::SymInt nsplit,
    at::Tensor& workspace, c10::SymInt max_rows) {
  const c10::DeviceGuard guard(q.device());
  const int64_t M = q.size(0), d = q.size(1);
  const int C = as_int(cmax), K = as_int(kk);
  at::Tensor w = at::empty({M, C}, f32(q)), idx = at::empty({M, K}, i32(q)), wsel = at::empty({M, K}, f32(q));
  at::Tensor r = at::empty({M, pages.size(-1)}, f32(q));
  if (M)
    check(xenc_route_read_decode(ptr<const float>(q), q.stride(0), (int)M, (int)d, ptr<const float>(S),
                                 pages.data_ptr(), (int)pages.size(1), pages.stride(0), ptr<const int>(chunk_page),
                                 ptr<const int>(chunk_nvalid), ptr<const int>(chunk_ptr), ptr<const int>(q_group),
                                 (int)chunk_ptr.numel() - 1, as_int(top_k), (float)route_temp, ptr<float>(w),
                                 w.stride(0), ptr<int>(idx), ptr<float>(wsel), K, (float)read_temp,
                                 softmax ? 1 : 0, as_int(nsplit), ptr<float>(r), r.stride(0), workspace.data_ptr(),
                                 (size_t)workspace.numel(), as_int(max_rows), stream_of(q)),
          "xenc_route_read_decode");
  return {w, idx, wsel, r};
}

int joint_dtype(const at::Tensor& k) {
  if (k.scalar_type() == at::kHalf) return 0;
  TORCH_CHECK_VALUE(k.scalar_type() == at::kBFloat16, "paged_decode_joint: pools must be fp16 or bf16");
  return 1;
}

void paged_decode_joint(const at::Tensor& q, const at::Tensor& op_k, const at::Tensor& op_v, const at::Tensor& op_bt,
                        const at::Tensor& op_len, const at::Tensor& own_k, const at::Tensor& own_v,
                        const at::Tensor& own_bt, const at::Tensor& own_len, double scale, c10::SymInt nsplit,
                        c10::SymInt chunk, at::Tensor& workspace, c10::SymInt max_n, at::Tensor& out) {
  const c10::DeviceGuard guard(q.device());
  const int64_t N = q.size(0), hq = q.size(1), d = q.size(2), hkv = op_k.size(2);
  if (N == 0) return;
  check(xenc_paged_decode_joint(joint_dtype(op_k), (int)N, (int)hq, (int)hkv, (int)d, q.data_ptr(), q.stride(0),
                                q.stride(1), op_k.data_ptr(), op_v.data_ptr(), op_k.stride(0), op_k.stride(1),
                                op_k.stride(2), (int)op_k.size(1), ptr<const int>(op_bt), op_bt.stride(0),
                                ptr<const int>(op_len), own_k.data_ptr(), own_v.data_ptr(), own_k.stride(0),
                                own_k.stride(1), own_k.stride(2), (int)own_k.size(1), ptr<const int>(own_bt),
                                own_bt.stride(0), ptr<const int>(own_len), (float)scale, as_int(nsplit),
                                as_int(chunk), ptr<float>(out), out.stride(0), out.stride(1), workspace.data_ptr(),
                                (size_t)workspace.numel(), as_int(max_n), stream_of(q)),
        "xenc_paged_decode_joint");
}

// ---- the read by entries (csrc/entries.hip).  Shared operands of its calls:
struct Entries {
  int M, d, kk, G, n_chunks, max_rows, tile_rows, slots, blocks;
  const int *row_ptr, *chunk_ptr, *list, *count, *chunk_page, *chunk_nvalid;
  void* st;
  float* stats = nullptr;   // [M kk][blocks] when a softmax page is read in several slot blocks

  void scores(int mode, const at::Tensor& x, const at::Tensor& pages_a, double temp, const at::Tensor* w,
              const at::Tensor& p, const at::Tensor* ds, const at::Tensor* gamma) const {
    check(xenc_entries_scores(mode, x.data_ptr(), M, d, kk, row_ptr, chunk_ptr, G, n_chunks, max_rows, list, count,
                              tile_rows, pages_a.data_ptr(), slots, pages_a.stride(0), chunk_page, chunk_nvalid,
                              (float)temp, w ? ptr<const float>(*w) : nullptr, w ? w->stride(0) : 0, p.data_ptr(),
                              ds ? ds->data_ptr() : nullptr, gamma ? ptr<float>(*gamma) : nullptr, blocks, stats, st),
          "xenc_entries_scores");
  }
  // out [M, d] = the readout of a [M kk, slots], scaled by w when given; idx NULL: rank j is chunk j.
  at::Tensor readout(const at::Tensor& a, const at::Tensor& pages_b, const at::Tensor* w, const int* idx,
                     const at::Tensor* route_w, const at::Tensor* gamma, const at::Tensor* dw_ext,
                     const at::Tensor* S, double route_temp) const {
    at::Tensor out = at::empty({M, d}, a.options().dtype(at::kFloat));
    const bool by_row = kk == 1 && !S;   // one entry a row: the readout writes the rows themselves
    at::Tensor part = by_row ? out : at::empty({(int64_t)M * kk, d}, out.options());
    check(xenc_entries_readout(a.data_ptr(), M, d, kk, row_ptr, chunk_ptr, G, n_chunks, max_rows, list, count,
                               tile_rows, pages_b.data_ptr(), slots, pages_b.stride(0), chunk_page,
                               w ? ptr<const float>(*w) : nullptr, w ? w->stride(0) : 0, by_row ? 1 : 0, blocks,
                               stats, ptr<float>(part), part.stride(0), st),
          "xenc_entries_readout");
    if (!by_row)
      check(xenc_entries_merge(ptr<const float>(part), M, d, kk, idx, row_ptr, chunk_ptr, G,
                               route_w ? ptr<const float>(*route_w) : nullptr, route_w ? route_w->stride(0) : 0,
                               gamma ? ptr<const float>(*gamma) : nullptr, dw_ext ? ptr<const float>(*dw_ext) : nullptr,
                               dw_ext ? dw_ext->stride(0) : 0, S ? ptr<const float>(*S) : nullptr, (float)route_temp,
                               ptr<float>(out), out.stride(0), st),
            "xenc_entries_merge");
    return out;
  }
};

at::Tensor rows_f16(const at::Tensor& x, void* st) {
  at::Tensor y = at::empty({x.size(0), x.size(1)}, x.options().dtype(at::kHalf));
  check(xenc_cast_rows_f16(ptr<const float>(x), x.stride(0), (int)x.size(0), (int)x.size(1), y.data_ptr(), st),
        "xenc_cast_rows_f16");
  return y;
}

at::Tensor read_entries(const at::Tensor& q, const at::Tensor& w, const c10::optional<at::Tensor>& idx,
                        const at::Tensor& frag_k_scores, const at::Tensor& frag_v_readout, const at::Tensor& chunk_ptr,
                        const at::Tensor& row_ptr, const at::Tensor& chunk_page, const at::Tensor& chunk_nvalid,
                        c10::SymInt max_rows, c10::SymInt tile_rows, c10::SymInt blocks, c10::SymInt slots,
                        double read_temp, bool softmax) {
  const c10::DeviceGuard guard(q.device());
  const int64_t M = q.size(0), d = q.size(1);
  if (M == 0) return at::empty({M, d}, f32(q));
  void* st = stream_of(q);
  Entries E{(int)M, (int)d, (int)(idx ? idx->size(1) : w.size(1)), (int)chunk_ptr.numel() - 1, (int)chunk_page.numel(),
            as_int(max_rows), as_int(tile_rows), as_int(slots), as_int(blocks), ptr<const int>(row_ptr),
            ptr<const int>(chunk_ptr), nullptr, nullptr, ptr<const int>(chunk_page), ptr<const int>(chunk_nvalid), st};
  at::Tensor list, count;
  if (idx) {
    list = at::empty({E.n_chunks, E.max_rows}, i32(q));
    count = at::empty({E.n_chunks}, i32(q));
    check(xenc_entries_list(ptr<const int>(*idx), E.M, E.kk, E.row_ptr, E.chunk_ptr, E.G, E.n_chunks, E.max_rows,
                            ptr<int>(list), ptr<int>(count), st),
          "xenc_entries_list");
    E.list = ptr<const int>(list);
    E.count = ptr<const int>(count);
  }
  at::Tensor p = at::empty({M * E.kk, E.slots}, q.options().dtype(at::kHalf)), stats;
  if (softmax && E.blocks > 1) {
    stats = at::empty({M * E.kk, E.blocks, 2}, f32(q));
    E.stats = ptr<float>(stats);
  }
  E.scores(softmax ? 0 : 2, rows_f16(q, st), frag_k_scores, read_temp, nullptr, p, nullptr, nullptr);
  return E.readout(p, frag_v_readout, &w, idx ? ptr<const int>(*idx) : nullptr, nullptr, nullptr, nullptr, nullptr, 0.);
}

std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor, at::Tensor, at::Tensor, at::Tensor> library_read_entries(
    const at::Tensor& q, const at::Tensor& S, const at::Tensor& chunk_ptr, const at::Tensor& row_ptr,
    const at::Tensor& logit_tiles, const at::Tensor& route_tiles, c10::SymInt n_logit, c10::SymInt n_route,
    c10::SymInt top_k, double route_temp, c10::SymInt cmax, c10::SymInt kk, const at::Tensor& frag_k_scores,
    const at::Tensor& frag_v_readout, const at::Tensor& frag_v_scores, const at::Tensor& frag_k_readout,
    const at::Tensor& chunk_page, const at::Tensor& chunk_nvalid, c10::SymInt max_rows, c10::SymInt tile_rows,
    c10::SymInt slots, double read_temp, bool softmax) {
  const c10::DeviceGuard guard(q.device());
  const int64_t M = q.size(0), d = q.size(1);
  void* st = stream_of(q);
  Entries E{(int)M, (int)d, as_int(kk), (int)chunk_ptr.numel() - 1, (int)chunk_page.numel(), as_int(max_rows),
            as_int(tile_rows), as_int(slots), 1, ptr<const int>(row_ptr), ptr<const int>(chunk_ptr), nullptr, nullptr,
            ptr<const int>(chunk_page), ptr<const int>(chunk_nvalid), st};
  at::Tensor w = at::empty({M, as_int(cmax)}, f32(q)), idx = at::empty({M, E.kk}, i32(q)),
             wsel = at::empty({M, E.kk}, f32(q)), qh = at::empty({M, d}, q.options().dtype(at::kHalf)),
             list = at::empty({E.n_chunks, E.max_rows}, i32(q)), count = at::empty({E.n_chunks}, i32(q)),
             p = at::empty({M * E.kk, E.slots}, qh.options());
  if (M == 0) return {at::empty({M, d}, f32(q)), w, idx, wsel, p, list, count.zero_()};
  check(xenc_route_topk_rows(ptr<const float>(q), q.stride(0), E.M, E.d, ptr<const float>(S), E.chunk_ptr, E.row_ptr,
                             ptr<const int>(logit_tiles), E.G, as_int(n_logit), as_int(top_k), (float)route_temp,
                             ptr<float>(w), w.stride(0), ptr<int>(idx), ptr<float>(wsel), E.kk, qh.data_ptr(), st),
        "xenc_route_topk_rows");
  check(xenc_entries_list(ptr<const int>(idx), E.M, E.kk, E.row_ptr, E.chunk_ptr, E.G, E.n_chunks, E.max_rows,
                          ptr<int>(list), ptr<int>(count), st),
        "xenc_entries_list");
  E.list = ptr<const int>(list);
  E.count = ptr<const int>(count);
  E.scores(softmax ? 0 : 2, qh, frag_k_scores, read_temp, nullptr, p, nullptr, nullptr);
  at::Tensor r = E.readout(p, frag_v_readout, &w, ptr<const int>(idx), nullptr, nullptr, nullptr, nullptr, 0.);
  return {r, w, idx, wsel, p, list, count};
}

using EntriesOut = std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor, at::Tensor, at::Tensor, at::Tensor>;

at::Tensor library_read_entries_bwd(const at::Tensor& g, const at::Tensor& w, const at::Tensor& idx,
                                    const at::Tensor& p, const c10::optional<at::Tensor>& dw_ext, const at::Tensor& S,
                                    const at::Tensor& list, const at::Tensor& count, const at::Tensor& frag_v_scores,
                                    const at::Tensor& frag_k_readout, const at::Tensor& chunk_ptr,
                                    const at::Tensor& chunk_page, const at::Tensor& chunk_nvalid,
                                    const at::Tensor& row_ptr, c10::SymInt max_rows, c10::SymInt tile_rows,
                                    c10::SymInt slots, double read_temp, bool softmax, double route_temp) {
  const c10::DeviceGuard guard(g.device());
  const int64_t M = g.size(0), d = g.size(1);
  if (M == 0) return at::empty({M, d}, f32(g));
  void* st = stream_of(g);
  const Entries E{(int)M, (int)d, (int)idx.size(1), (int)chunk_ptr.numel() - 1, (int)chunk_page.numel(),
                  as_int(max_rows), as_int(tile_rows), as_int(slots), 1, ptr<const int>(row_ptr),
                  ptr<const int>(chunk_ptr), ptr<const int>(list), ptr<const int>(count), ptr<const int>(chunk_page),
                  ptr<const int>(chunk_nvalid), st};
  at::Tensor ds = at::empty_like(p), gamma = at::empty({M * E.kk}, f32(g));
  E.scores(softmax ? 1 : 3, rows_f16(g, st), frag_v_scores, read_temp, &w, p, &ds, &gamma);
  return E.readout(ds, frag_k_readout, nullptr, ptr<const int>(idx), &w, &gamma, dw_ext ? &*dw_ext : nullptr, &S,
                   route_temp);
}

// Autograd of library_read_entries.  Both directions go through the dispatcher (fake tensors and
// functionalisation see the two operators); no gradient is materialised for the outputs nothing
// differentiates.
class EntriesRead : public torch::autograd::Function<EntriesRead> {
 public:
  static torch::autograd::variable_list forward(
      torch::autograd::AutogradContext* ctx, const at::Tensor& q, const at::Tensor& S, const at::Tensor& chunk_ptr,
      const at::Tensor& row_ptr, const at::Tensor& logit_tiles, const at::Tensor& route_tiles, c10::SymInt n_logit,
      c10::SymInt n_route, c10::SymInt top_k, double route_temp, c10::SymInt cmax, c10::SymInt kk,
      const at::Tensor& frag_k_scores, const at::Tensor& frag_v_readout, const at::Tensor& frag_v_scores,
      const at::Tensor& frag_k_readout, const at::Tensor& chunk_page, const at::Tensor& chunk_nvalid,
      c10::SymInt max_rows, c10::SymInt tile_rows, c10::SymInt slots, double read_temp, bool softmax) {
    at::AutoDispatchBelowADInplaceOrView guard;
    static const auto op = c10::Dispatcher::singleton()
                               .findSchemaOrThrow("xenc::library_read_entries", "")
                               .typed<decltype(library_read_entries)>();
    auto [r, w, idx, wsel, p, list, count] =
        op.call(q, S, chunk_ptr, row_ptr, logit_tiles, route_tiles, n_logit, n_route, top_k, route_temp, cmax, kk,
                frag_k_scores, frag_v_readout, frag_v_scores, frag_k_readout, chunk_page, chunk_nvalid, max_rows,
                tile_rows, slots, read_temp, softmax);
    ctx->save_for_backward({w, idx, p, list, count, frag_v_scores, frag_k_readout, chunk_ptr, chunk_page, chunk_nvalid,
                            row_ptr, S, route_tiles});
    ctx->saved_data["n_route"] = n_route;
    ctx->saved_data["max_rows"] = max_rows;
    ctx->saved_data["tile_rows"] = tile_rows;
    ctx->saved_data["slots"] = slots;
    ctx->saved_data["d"] = q.sym_size(1);
    ctx->saved_data["read_temp"] = read_temp;
    ctx->saved_data["route_temp"] = route_temp;
    ctx->saved_data["softmax"] = softmax;
    ctx->mark_non_differentiable({idx, wsel, p, list, count});
    ctx->set_materialize_grads(false);
    return {r, w, idx, wsel, p, list, count};
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const auto v = ctx->get_saved_variables();
    const at::Tensor &w = v[0], &idx = v[1], &p = v[2], &list = v[3], &count = v[4], &fvs = v[5], &fkr = v[6],
                     &chunk_ptr = v[7], &chunk_page = v[8], &chunk_nvalid = v[9], &row_ptr = v[10], &S = v[11],
                     &route_tiles = v[12];
    auto& sd = ctx->saved_data;
    const at::Tensor &dr = grads[0], &dw = grads[1];
    const double route_temp = sd["route_temp"].toDouble();
    c10::optional<at::Tensor> dwc;
    if (dw.defined()) dwc = dw.contiguous();
    at::Tensor dq;
    if (dr.defined()) {
      static const auto op = c10::Dispatcher::singleton()
                                 .findSchemaOrThrow("xenc::library_read_entries_bwd", "")
                                 .typed<decltype(library_read_entries_bwd)>();
      dq = op.call(dr.contiguous(), w, idx, p, dwc, S, list, count, fvs, fkr, chunk_ptr, chunk_page, chunk_nvalid,
                   row_ptr, sd["max_rows"].toSymInt(), sd["tile_rows"].toSymInt(), sd["slots"].toSymInt(),
                   sd["read_temp"].toDouble(), sd["softmax"].toBool(), route_temp);
    } else {   // only w reaches the loss: the routing term alone (nothing at all: 0)
      dq = at::zeros_symint({w.sym_size(0), sd["d"].toSymInt()}, w.options());
      if (dwc) {
        static const auto op = c10::Dispatcher::singleton()
                                   .findSchemaOrThrow("xenc::route_backward_", "")
                                   .typed<void(at::Tensor&, const at::Tensor&, const at::Tensor&,
                                               const c10::optional<at::Tensor>&, const at::Tensor&, const at::Tensor&,
                                               const at::Tensor&, const at::Tensor&, c10::SymInt, double)>();
        op.call(dq, w, at::zeros_like(w), dwc, S, chunk_ptr, row_ptr, route_tiles, sd["n_route"].toSymInt(), route_temp);
      }
    }
    torch::autograd::variable_list out(23);
    out[0] = dq;
    return out;
  }
};

EntriesOut library_read_entries_autograd(
    const at::Tensor& q, const at::Tensor& S, const at::Tensor& chunk_ptr, const at::Tensor& row_ptr,
    const at::Tensor& logit_tiles, const at::Tensor& route_tiles, c10::SymInt n_logit, c10::SymInt n_route,
    c10::SymInt top_k, double route_temp, c10::SymInt cmax, c10::SymInt kk, const at::Tensor& frag_k_scores,
    const at::Tensor& frag_v_readout, const at::Tensor& frag_v_scores, const at::Tensor& frag_k_readout,
    const at::Tensor& chunk_page, const at::Tensor& chunk_nvalid, c10::SymInt max_rows, c10::SymInt tile_rows,
    c10::SymInt slots, double read_temp, bool softmax) {
  auto o = EntriesRead::apply(q, S, chunk_ptr, row_ptr, logit_tiles, route_tiles, n_logit, n_route, top_k, route_temp,
                              cmax, kk, frag_k_scores, frag_v_readout, frag_v_scores, frag_k_readout, chunk_page,
                              chunk_nvalid, max_rows, tile_rows, slots, read_temp, softmax);
  return {o[0], o[1], o[2], o[3], o[4], o[5], o[6]};
}

// ---- a hooked layer around its read (xenc/injector.py:54-77, 185-197)
// (hn, q) of rows h [M, d_m]: hn = rms_norm(h), q = A hn / (|A hn| + eps).
std::tuple<at::Tensor, at::Tensor> hook_query(const at::Tensor& h, const at::Tensor& A,
                                              const c10::optional<at::Tensor>& bias, double eps) {
  const c10::DeviceGuard guard(h.device());
  void* st = stream_of(h);
  at::Tensor hn = at::empty({h.size(0), h.size(1)}, f32(h));
  check(xenc_hook_norm(ptr<const float>(h), h.stride(0), (int)h.size(0), (int)h.size(1), (float)eps, ptr<float>(hn), st),
        "xenc_hook_norm");
  at::Tensor q = at::linear(hn, A, bias);
  check(xenc_hook_unit(ptr<float>(q), q.stride(0), (int)q.size(0), (int)q.size(1), (float)eps, st), "xenc_hook_unit");
  return {hn, q};
}

// delta [M, d_out] = scale * (W r + bias), scale = gain_scale exp(log_gain) sigmoid(hn . gate_w + gate_b).
at::Tensor hook_write(const at::Tensor& hn, const at::Tensor& r, const at::Tensor& gate_w, const at::Tensor& gate_b,
                      const at::Tensor& log_gain, double gain_scale, const at::Tensor& W,
                      const c10::optional<at::Tensor>& bias) {
  const c10::DeviceGuard guard(r.device());
  void* st = stream_of(r);
  const int M = (int)r.size(0), d = (int)r.size(1), d_out = (int)W.size(0);
  at::Tensor scale = at::empty({M}, f32(r)), out = at::empty({M, d_out}, f32(r));
  check(xenc_gate_scale(M, (int)hn.size(1), ptr<const float>(hn), hn.stride(0), nullptr, nullptr, 1,
                        ptr<const float>(gate_w), ptr<const float>(gate_b), ptr<const float>(log_gain),
                        (float)gain_scale, ptr<float>(scale), st),
        "xenc_gate_scale");
  check(xenc_write_back(ptr<const float>(r), r.stride(0), M, d, nullptr, 1, ptr<const float>(W),
                        (long long)d_out * W.stride(0), W.stride(0), d_out, bias ? ptr<const float>(*bias) : nullptr, 0,
                        ptr<const float>(scale), ptr<float>(out), out.stride(0), st),
        "xenc_write_back");
  return out;
}

// (h + delta, |delta| / (|h| + 1e-6) per row) of rows h, delta [M, d].
std::tuple<at::Tensor, at::Tensor> hook_add(const at::Tensor& h, const at::Tensor& delta) {
  const c10::DeviceGuard guard(h.device());
  at::Tensor out = at::empty({h.size(0), h.size(1)}, f32(h)), ratio = at::empty({h.size(0)}, f32(h));
  check(xenc_hook_add(ptr<const float>(h), h.stride(0), ptr<const float>(delta), delta.stride(0), (int)h.size(0),
                      (int)h.size(1), ptr<float>(out), ptr<float>(ratio), stream_of(h)),
        "xenc_hook_add");
  return {out, ratio};
}

// One hooked layer of a decode step over one library, rows h [M, d_m]: hook_query, route_read (rows of one
// library), hook_write and hook_add in one call, the same launches and bits.  maps = (A, gate_w, gate_b,
// log_gain, B), pool = (S, pages, chunk_page, chunk_nvalid, chunk_ptr); sizes = (position of the layer in
// gate_b / log_gain, top_k, cmax, kk, nsplit, workspace rows), scales = (eps, gain, route_temp, read_temp).
// -> (h + delta, w [M, cmax], mean of |delta| / |h|).
std::tuple<at::Tensor, at::Tensor, at::Tensor> hook_layer(const at::Tensor& h, at::TensorList maps,
                                                          const c10::optional<at::Tensor>& a_bias,
                                                          const c10::optional<at::Tensor>& b_bias, at::TensorList pool,
                                                          c10::IntArrayRef sizes, c10::ArrayRef<double> scales,
                                                          bool softmax, at::Tensor& workspace) {
  TORCH_CHECK_VALUE(maps.size() == 5 && pool.size() == 5 && sizes.size() == 6 && scales.size() == 4,
                    "hook_layer: 5 maps, 5 pool tensors, 6 sizes and 4 scales");
  const c10::DeviceGuard guard(h.device());
  auto [hn, q] = hook_query(h, maps[0], a_bias, scales[0]);
  const at::Tensor group = at::zeros({h.size(0)}, i32(h));
  auto [w, idx, wsel, r] = route_read(q, pool[0], pool[1], pool[2], pool[3], pool[4], group, sizes[1], scales[2], sizes[2],
                                      sizes[3], scales[3], softmax, sizes[4], workspace, sizes[5]);
  const int64_t p = sizes[0];
  const at::Tensor delta = hook_write(hn, r, maps[1], maps[2].slice(0, p, p + 1), maps[3].slice(0, p, p + 1), scales[1],
                                      maps[4], b_bias);
  auto [out, ratio] = hook_add(h, delta);
  return {out, w, ratio.mean()};
}

}  // namespace

TORCH_LIBRARY_FRAGMENT(xenc, m) {
  m.def("route_topk(Tensor q, Tensor S, Tensor chunk_ptr, Tensor q_group, SymInt top_k, float route_temp, "
        "SymInt cmax, SymInt kk) -> (Tensor, Tensor, Tensor)");
  m.def("library_read(Tensor q, Tensor pages, Tensor chunk_page, Tensor chunk_nvalid, Tensor chunk_ptr, "
        "Tensor q_group, Tensor idx, Tensor w_sel, float read_temp, bool softmax, SymInt nsplit, "
        "Tensor(a!) workspace, SymInt max_rows) -> Tensor");
  m.def("route_read(Tensor q, Tensor S, Tensor pages, Tensor chunk_page, Tensor chunk_nvalid, Tensor chunk_ptr, "
        "Tensor q_group, SymInt top_k, float route_temp, SymInt cmax, SymInt kk, float read_temp, bool softmax, "
        "SymInt nsplit, Tensor(a!) workspace, SymInt max_rows) -> (Tensor, Tensor, Tensor, Tensor)");
  m.def("paged_decode_joint(Tensor q, Tensor op_k, Tensor op_v, Tensor op_bt, Tensor op_len, Tensor own_k, "
        "Tensor own_v, Tensor own_bt, Tensor own_len, float scale, SymInt nsplit, SymInt chunk, "
        "Tensor(a!) workspace, SymInt max_n, Tensor(b!) out) -> ()");
  m.def("hook_query(Tensor h, Tensor A, Tensor? bias, float eps) -> (Tensor, Tensor)");
  m.def("hook_write(Tensor hn, Tensor r, Tensor gate_w, Tensor gate_b, Tensor log_gain, float gain_scale, Tensor W, "
        "Tensor? bias) -> Tensor");
  m.def("hook_add(Tensor h, Tensor delta) -> (Tensor, Tensor)");
  m.def("hook_layer(Tensor h, Tensor[] maps, Tensor? a_bias, Tensor? b_bias, Tensor[] pool, int[] sizes, "
        "float[] scales, bool softmax, Tensor(a!) workspace) -> (Tensor, Tensor, Tensor)");
  m.def("read_entries(Tensor q, Tensor w, Tensor? idx, Tensor frag_k_scores, Tensor frag_v_readout, Tensor chunk_ptr, "
        "Tensor row_ptr, Tensor chunk_page, Tensor chunk_nvalid, SymInt max_rows, SymInt tile_rows, SymInt blocks, "
        "SymInt slots, float read_temp, bool softmax) -> Tensor");
  m.def("library_read_entries(Tensor q, Tensor S, Tensor chunk_ptr, Tensor row_ptr, Tensor logit_tiles, "
        "Tensor route_tiles, SymInt n_logit, SymInt n_route, SymInt top_k, float route_temp, SymInt cmax, SymInt kk, "
        "Tensor frag_k_scores, Tensor frag_v_readout, Tensor frag_v_scores, Tensor frag_k_readout, Tensor chunk_page, "
        "Tensor chunk_nvalid, SymInt max_rows, SymInt tile_rows, SymInt slots, float read_temp, bool softmax) -> "
        "(Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor)");
  m.def("library_read_entries_bwd(Tensor g, Tensor w, Tensor idx, Tensor p, Tensor? dw_ext, Tensor S, Tensor list, "
        "Tensor count, Tensor frag_v_scores, Tensor frag_k_readout, Tensor chunk_ptr, Tensor chunk_page, "
        "Tensor chunk_nvalid, Tensor row_ptr, SymInt max_rows, SymInt tile_rows, SymInt slots, float read_temp, "
        "bool softmax, float route_temp) -> Tensor");
}

TORCH_LIBRARY_IMPL(xenc, Autograd, m) { m.impl("library_read_entries", &library_read_entries_autograd); }

TORCH_LIBRARY_IMPL(xenc, CUDA, m) {
  m.impl("route_topk", &route_topk);
  m.impl("library_read", &library_read);
  m.impl("route_read", &route_read);
  m.impl("paged_decode_joint", &paged_decode_joint);
  m.impl("hook_query", &hook_query);
  m.impl("hook_write", &hook_write);
  m.impl("hook_add", &hook_add);
  m.impl("hook_layer", &hook_layer);
  m.impl("read_entries", &read_entries);
  m.impl("library_read_entries", &library_read_entries);
  m.impl("library_read_entries_bwd", &library_read_entries_bwd);
}
