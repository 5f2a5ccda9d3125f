/*
 * hcs_noalloc.hip -- a contact step that allocates nothing
 * (hcs_contact_step_noalloc).  No reference counterpart: it is
 * hcs_contact_step for callers that cannot allocate device memory (code
 * under HIP graph capture, tight serving loops, hosts that forbid
 * hipMalloc).
 *
 * Every device buffer of the step (env descriptors, state, work items, the
 * pipeline's counters, survivors, contributions, scan storage, reduction
 * partials and per-pair outputs) is a slice of one file-scope array, `scratch`,
 * of HCS_SCRATCH_BYTES + HCS_SCRATCH_EXTRA on each device.  Its device address
 * comes from hipGetSymbolAddress, taken once per device with that device
 * current (hcs_create calls scratch_setup); host code only ever uses that
 * address.  The slices are laid out per call from the call's
 * sizes; a call that does not fit returns HCS_ERR_CAPACITY before anything
 * runs, or (survivors beyond the space left) after the step with every
 * pair's counts valid and its status HCS_ERR_CAPACITY.
 *
 * The array is shared by every call on one device and keeps the last call's
 * contents; every counter is cleared by a fill kernel at the start of each
 * step.  Calls that overlap on one device (two contexts, two host threads)
 * race on it.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "hcs_internal.h"
#include "hcs_prim.h"

/* What a call may use: 64 MiB per device, room for about 690k survivors of
 * the exact rejections after the per-call tables of a few hundred pairs.  The
 * array holds a little more: the work items of the engine's own splitting (at
 * most its item budget, 44 bytes each) are not the caller's to pay for. */
#define HCS_SCRATCH_BYTES (64ull << 20)
#define HCS_SCRATCH_EXTRA (4ull << 20)

static __device__ __align__(256) unsigned char scratch[HCS_SCRATCH_BYTES + HCS_SCRATCH_EXTRA];

namespace hcs {

namespace {
std::mutex g_scratch_mu;
/* per device ordinal: the device address of `scratch` (nullptr: not yet) */
std::vector<void*> g_scratch_ptr;
}  // namespace

int scratch_setup(Ctx* c) {
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if ((int)g_scratch_ptr.size() <= c->device) g_scratch_ptr.resize(c->device + 1, nullptr);
  if (!g_scratch_ptr[c->device]) {
    int cur = -1;
    hipError_t e = hipGetDevice(&cur);
    if (e == hipSuccess && cur != c->device) e = hipSetDevice(c->device);
    void* p = nullptr;
    if (e == hipSuccess) e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) return hip_check(c, e == hipSuccess ? hipErrorInvalidSymbol : e, "hipGetSymbolAddress");
    g_scratch_ptr[c->device] = p;
  }
  c->scratch = g_scratch_ptr[c->device];
  c->scratch_bytes = HCS_SCRATCH_BYTES + HCS_SCRATCH_EXTRA;
  return HCS_OK;
}

namespace {

/* Carves 256-byte-aligned fixed slices off the scratch array. */
struct Carver {
  unsigned char* base;
  size_t size, used = 0;
  bool ok = true;
  void take(DBuf& b, size_t bytes) {
    bytes = std::max<size_t>(bytes, 8);
    const size_t at = (used + 255) & ~(size_t)255;
    b.fixed = true;
    if (at + bytes > size) {
      ok = false;
      b.ptr = nullptr, b.bytes = 0;
      return;
    }
    b.ptr = base + at, b.bytes = bytes;
    used = at + bytes;
  }
  size_t left() const { return size > ((used + 255) & ~(size_t)255) ? size - ((used + 255) & ~(size_t)255) : 0; }
};

/* Survivors a call may have, by a fixed price list: bytes per pair, work item
 * (64 queries, unsplit), moved triangle and reduction slice (8 items, at most
 * 64 per pair), slices of 256 bytes, the rest 96 bytes per survivor.  Which
 * calls fit is thus a matter of their sizes, whatever tables the engine keeps
 * for them.  Negative: the tables alone do not fit. */
int64_t admitted_survivors(const Plan& plan) {
  const size_t np = plan.envs.size();
  size_t ni = 0, slices = 0;
  for (const EnvDesc& E : plan.envs) {
    const size_t n = (size_t)(E.item_count >> E.depth);
    ni += n;
    slices += std::max<size_t>(1, std::min<size_t>(64, (n + 7) / 8));
  }
  ni = std::max<size_t>(1, ni);
  size_t used = 0;
  auto take = [&](size_t bytes) { used = ((used + 255) & ~(size_t)255) + std::max<size_t>(bytes, 8); };
  for (size_t per : {184, 288}) take(per * np);
  take(16 * ni);
  for (int k = 0; k < 3; ++k) take(64);
  take(96 * np), take(4 * ni), take(4 * (ni + 1)), take(4 * (ni + 1)), take(128 * np);
  take(scan_temp_bytes((long long)ni + 1));
  take(96 * ni), take(4 * ni), take(16 * ni), take(36);
  take(144 * (size_t)std::max<int64_t>(1, plan.ntx)), take(4 * std::max<size_t>(1, plan.xenv.size())), take(8);
  take(16 * slices), take(8 * np), take(672 * slices);
  used = (used + 255) & ~(size_t)255;
  if (used + 512 > HCS_SCRATCH_BYTES) return -1;
  return (int64_t)((HCS_SCRATCH_BYTES - used - 512) / (sizeof(int4) + sizeof(Contrib)));
}

}  // namespace

}  // namespace hcs

using namespace hcs;

extern "C" int hcs_contact_step_noalloc(hcs_ctx* h, int32_t npairs, const hcs_pair_in* in, const hcs_step_opts* opts,
                                        hcs_pair_out* out) {
  if (!h || npairs < 0 || (npairs > 0 && (!in || !out))) return HCS_ERR_ARG;
  Ctx* c = &h->c;
  if (opts && opts->keep_polygons)
    return set_err(c, HCS_ERR_ARG, "hcs_contact_step_noalloc keeps no polygons (keep_polygons must be 0)");
  if (!c->scratch) return set_err(c, HCS_ERR_STATE, "scratch array not set up on this device");
  if (npairs == 0) return HCS_OK;
  int rc = hip_check(c, hipSetDevice(c->device), "hipSetDevice");
  if (rc) return rc;
  /* the plan on the host, then the slices for its sizes */
  std::vector<int32_t> geoms(2 * (size_t)npairs);
  for (int e = 0; e < npairs; ++e) geoms[2 * e] = in[e].geom_a, geoms[2 * e + 1] = in[e].geom_b;
  Plan plan;
  if ((rc = build_plan(c, npairs, geoms.data(), opts, c->tet_mode_max_tris, plan, ITEMS_IMPLICIT))) return rc;
  const int64_t cap = admitted_survivors(plan);
  if (cap < 4096) {
    size_t items = 0;
    for (const EnvDesc& E : plan.envs) items += (size_t)(E.item_count >> E.depth);
    return set_err(c, HCS_ERR_CAPACITY,
                   "hcs_contact_step_noalloc: " + std::to_string(npairs) + " pairs and " + std::to_string(items) +
                       " work items do not fit the " + std::to_string(HCS_SCRATCH_BYTES >> 20) + " MiB scratch array");
  }
  CallBlob blob;
  const CallSizes z = call_sizes(plan);
  const size_t np = npairs, nb = z.blocks1 + z.blocks2;
  const size_t blob_bytes = call_blob_bytes(plan, blob), out_bytes = sizeof(PairOut) * np + sizeof(CallTail);
  Carver cv{(unsigned char*)c->scratch, c->scratch_bytes};
  Pipe P;
  cv.take(P.blob, blob_bytes);
  cv.take(P.counter, 64);
  cv.take(P.surv_cnt, 64);
  cv.take(P.err, 64);
  cv.take(P.xf, sizeof(double) * 12 * np);
  cv.take(P.xtri, sizeof(double) * HCS_XTRI * std::max<int64_t>(1, plan.ntx));
  cv.take(P.gen_cnt, sizeof(unsigned) * (nb + 1));
  cv.take(P.gen_mask, sizeof(unsigned long long) * nb * (HCS_GEN_THREADS / 64));
  cv.take(P.gen_item, sizeof(int4) * z.items);
  cv.take(P.pair_lo, sizeof(int) * (np + 1));
  cv.take(P.live_item, sizeof(int4) * z.live);
  cv.take(P.ncand, sizeof(int) * z.live);
  cv.take(P.nsurv, sizeof(unsigned) * (z.live + 1));
  cv.take(P.off, sizeof(unsigned) * (z.live + 1));
  cv.take(P.scan_tmp, scan_temp_bytes((long long)z.live + 1));
  cv.take(P.part, sizeof(RedPart) * np * z.slices);
  cv.take(P.out, out_bytes);
  cv.take(P.surv, sizeof(int4) * cap);
  cv.take(P.contrib, sizeof(Contrib) * cap);
  if (!cv.ok) return set_err(c, HCS_ERR_CAPACITY, "hcs_contact_step_noalloc: scratch layout");
  /* every request below fits its slice (ensure() on a fixed slice never
   * allocates and reports anything larger as HCS_ERR_CAPACITY) */
  if ((rc = call_reserve(c, P, plan, blob, cap))) return rc;
  /* the blob goes through the context's pinned memory as long as that holds
   * it (it is not grown here), else by a copy from ordinary memory */
  std::vector<char> image;
  if (blob_bytes <= c->pin_up_bytes) {
    call_blob_fill(plan, in, blob, (char*)c->pin_up);
    blob.src = c->pin_up;
  } else {
    image.resize(blob_bytes);
    call_blob_fill(plan, in, blob, image.data());
    rc = hip_check(c, hipMemcpyAsync(P.blob.ptr, image.data(), blob_bytes, hipMemcpyHostToDevice, c->stream), "upload");
    if (rc) return rc;
    blob.src = P.blob.ptr;
  }
  const bool direct = out_bytes <= c->pin_down_bytes;
  char* down = direct ? (char*)c->pin_down : (char*)P.out.ptr;
  CallTail tail{};
  QueryArgs a = call_args(P, plan, blob);
  if ((rc = call_enqueue(c, P, a, plan, blob, nullptr, 0, false, c->num_cu * 12, (PairOut*)down,
                         (CallTail*)(down + sizeof(PairOut) * np))))
    return rc;
  rc = hip_check(c, hipGetLastError(), "noalloc step");
  static_assert(sizeof(hcs_pair_out) == sizeof(PairOut), "pair_out layout");
  if (!rc && !direct)
    rc = hip_check(c, hipMemcpyAsync(out, down, sizeof(PairOut) * np, hipMemcpyDeviceToHost, c->stream), "dl");
  if (!rc && !direct)
    rc = hip_check(c, hipMemcpyAsync(&tail, down + sizeof(PairOut) * np, sizeof tail, hipMemcpyDeviceToHost, c->stream),
                   "dl");
  if (!rc) rc = hip_check(c, hipStreamSynchronize(c->stream), "sync");
  if (rc) return rc;
  if (direct) {
    std::memcpy(out, down, sizeof(PairOut) * np);
    std::memcpy(&tail, down + sizeof(PairOut) * np, sizeof tail);
  }
  if (tail.err) return set_err(c, HCS_ERR_LIMIT, "traversal stack overflow");
  if ((int64_t)tail.nsurv > P.cap)
    return set_err(c, HCS_ERR_CAPACITY, "hcs_contact_step_noalloc: " + std::to_string(tail.nsurv) +
                                            " survivors exceed the scratch array's room for " +
                                            std::to_string(P.cap));
  return HCS_OK;
}
