// kad_run_calls: a layer's launches, prepared once as argument structs, in one host call; kad_find_relocs:
// which of the structs' pointers move with the caller's tensors.
#include <string.h>

#include "kad_common.h"

using namespace kad;

namespace {
constexpr int64_t BLOB_MAX = 16384;

int64_t arg_size(int fn) {
  switch (fn) {
    case KAD_CALL_PYRAMID: return sizeof(kad_pyramid_args);
    case KAD_CALL_LCSA_PREP:
    case KAD_CALL_LCSA_MASK: return sizeof(kad_lcsa_args);
    case KAD_CALL_DSC: return sizeof(kad_dcn_args);
    case KAD_CALL_MERGE: return sizeof(kad_merge_args);
    case KAD_CALL_SCALE_RESIDUAL: return sizeof(kad_scale_args);
    default: return -1;
  }
}
}  // namespace

extern "C" int kad_run_calls(const void* blob, int64_t blob_bytes, const kad_call* calls, int ncalls,
                             const kad_reloc* relocs, int nrelocs, void* const* bases, int nbases, void* stream) {
  KAD_CHECK_ARG(blob && calls && (relocs || nrelocs == 0) && (bases || nbases == 0), "kad_run_calls: null pointer");
  KAD_CHECK_ARG(blob_bytes >= 0 && blob_bytes <= BLOB_MAX && ncalls >= 0 && nrelocs >= 0,
                "kad_run_calls: blob of %lld bytes, %d calls, %d relocations", (long long)blob_bytes, ncalls, nrelocs);
  alignas(16) unsigned char buf[BLOB_MAX];
  memcpy(buf, blob, (size_t)blob_bytes);
  for (int i = 0; i < nrelocs; ++i) {
    const kad_reloc& r = relocs[i];
    KAD_CHECK_ARG(r.at >= 0 && r.at % 8 == 0 && r.at + 8 <= blob_bytes && r.base >= 0 && r.base < nbases,
                  "kad_run_calls: relocation %d out of range", i);
    const uintptr_t p = (uintptr_t)bases[r.base] + (uintptr_t)r.add;
    memcpy(buf + r.at, &p, sizeof(p));
  }
  for (int i = 0; i < ncalls; ++i) {
    const kad_call& c = calls[i];
    const int64_t size = arg_size(c.fn);
    KAD_CHECK_ARG(size > 0 && c.count >= 1 && c.count <= BLOB_MAX / size && c.args >= 0 && c.args % 8 == 0 &&
                      c.args + size * c.count <= blob_bytes,
                  "kad_run_calls: call %d out of range", i);
    const void* a = buf + c.args;
    int rc = KAD_EINVAL;
    switch (c.fn) {
      case KAD_CALL_PYRAMID: rc = kad_pyramid_proj((const kad_pyramid_args*)a, stream); break;
      case KAD_CALL_LCSA_PREP: rc = kad_lcsa_prep_group((const kad_lcsa_args*)a, c.count, stream); break;
      case KAD_CALL_LCSA_MASK: rc = kad_lcsa_mask_group((const kad_lcsa_args*)a, c.count, c.arg, stream); break;
      case KAD_CALL_DSC: rc = kad_dsc_fwd_group((const kad_dcn_args*)a, c.count, stream); break;
      case KAD_CALL_MERGE: rc = kad_branch_merge((const kad_merge_args*)a, stream); break;
      case KAD_CALL_SCALE_RESIDUAL: {
        const kad_scale_args* s = (const kad_scale_args*)a;
        rc = kad_scale_residual(s->out, s->att, s->residual, s->n, s->c, s->h, s->w, s->img_c, s->c_off, s->layout,
                                s->dtype, stream);
        break;
      }
    }
    if (rc) return rc;
  }
  return KAD_OK;
}

extern "C" int kad_find_relocs(const void* blob, int64_t blob_bytes, const int64_t* at, int nat, const kad_span* spans,
                               int nspans, kad_reloc* relocs) {
  KAD_CHECK_ARG((blob || blob_bytes == 0) && (at || nat == 0) && (spans || nspans == 0) && (relocs || nat == 0),
                "kad_find_relocs: null pointer");
  KAD_CHECK_ARG(blob_bytes >= 0 && nat >= 0 && nspans >= 0, "kad_find_relocs: negative count");
  int n = 0;
  for (int i = 0; i < nat; ++i) {
    KAD_CHECK_ARG(at[i] >= 0 && at[i] + 8 <= blob_bytes, "kad_find_relocs: pointer %d outside the blob", i);
    int64_t p;
    memcpy(&p, (const char*)blob + at[i], sizeof(p));
    if (!p) continue;
    int start = 0, inside = 0;  // spans that begin at p, that hold it
    const kad_span *s0 = nullptr, *s1 = nullptr;
    for (int k = 0; k < nspans; ++k) {
      const kad_span& s = spans[k];
      if (p == s.ptr && s.bytes > 0) {
        ++start;
        s0 = &s;
      } else if (p > s.ptr && p < s.ptr + s.bytes) {
        ++inside;
        s1 = &s;
      }
    }
    // two channel slices of one buffer span each other's starts: a start decides
    KAD_CHECK_ARG(start <= 1 && (start == 1 || inside <= 1), "kad_find_relocs: pointer %d fits two spans", i);
    const kad_span* s = start ? s0 : s1;
    if (s) relocs[n++] = {at[i], s->off + (p - s->ptr), (int)s->base};
  }
  return n;
}
