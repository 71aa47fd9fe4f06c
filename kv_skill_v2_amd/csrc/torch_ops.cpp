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
//   xenc::library_read_entries, library_read_entries_bwd   routing + that read, and its dQ (autograd
//                             registered in torch_ops.py)
//   xenc::paged_decode_joint  DecodeReader.__call__ (xenc/d23_read_kernels.py:145-160)
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
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

TORCH_LIBRARY_IMPL(xenc, CUDA, m) {
  m.impl("route_topk", &route_topk);
  m.impl("library_read", &library_read);
  m.impl("route_read", &route_read);
  m.impl("paged_decode_joint", &paged_decode_joint);
  m.impl("read_entries", &read_entries);
  m.impl("library_read_entries", &library_read_entries);
  m.impl("library_read_entries_bwd", &library_read_entries_bwd);
}
