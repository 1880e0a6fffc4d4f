// The voxelizer's host side against a stand-in for the device: memory is host memory filled with
// garbage, allocations fail on demand, and the few kernels that matter here are imitated (fills,
// read-backs, and which buffers a pass leaves marked or clears). Checked at every mark kernel: the
// table, flags, cells and slots that it is given lie in live allocations and are zero; and at
// every launch, that the grid is one HIP accepts and that no argument points into memory that was
// given back (whose addresses are not used again here).
#include "../../ooc_svo_builder_amd/csrc/svo_voxelize.hip"

#include <sys/mman.h>

#include <cstdlib>
#include <map>
#include <string>

#include "../../include/svo_amd.h"

using namespace svo;

namespace {
constexpr size_t kHuge = 256u << 20;  // allocations above are address space, neither filled nor read
struct Device {
  std::map<uintptr_t, size_t> mem, gone;     // live allocations, those given back
  std::map<const void*, std::string> names;  // kernels
  long allocs = 0, fail_at = -1;             // allocations since arming; the one that fails
  uint64_t n_occ = 0, n_vox = 0;             // what a pass is said to find
  uint64_t found = 0;                        // its bricks: no more than there are
  uint64_t unclean = 0, outside = 0, bad_grid = 0, marks = 0, dense = 0, stale = 0;
  std::vector<uint8_t> args;  // of the launch (the library's launch log)
  hipError_t last = hipSuccess;
};
Device& dev() {
  static Device* d = new Device();
  return *d;
}
bool inside(const void* p, size_t bytes) {
  auto& m = dev().mem;
  auto it = m.upper_bound((uintptr_t)p);
  if (it == m.begin()) return bytes == 0;
  --it;
  return (uintptr_t)p + bytes <= it->first + it->second;
}
hipError_t allocate(void** p, size_t bytes) {
  Device& d = dev();
  *p = nullptr;
  if (d.allocs++ == d.fail_at) return d.last = hipErrorOutOfMemory;
  *p = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (bytes <= kHuge) memset(*p, 0xA5, bytes);
  d.mem[(uintptr_t)*p] = bytes;
  return hipSuccess;
}
hipError_t give_back(void* p) {
  Device& d = dev();
  const size_t bytes = d.mem[(uintptr_t)p];
  d.mem.erase((uintptr_t)p);
  // the addresses stay taken
  mmap(p, bytes, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE | MAP_FIXED, -1, 0);
  d.gone[(uintptr_t)p] = bytes;
  return hipSuccess;
}
// the launch's arguments, word by word: an address in memory that was given back
void look_for_stale() {
  Device& d = dev();
  for (size_t k = 0; k + 8 <= d.args.size(); k += 4) {
    uintptr_t v;
    memcpy(&v, d.args.data() + k, 8);
    auto it = d.gone.upper_bound(v);
    if (it == d.gone.begin()) continue;
    --it;
    if (v < it->first + it->second) d.stale++;
  }
  d.args.clear();
}
void must_be_zero(const void* p, size_t bytes) {
  if (!inside(p, bytes)) {
    dev().outside++;
    return;
  }
  if (bytes > kHuge) return;
  for (size_t k = 0; k < bytes; k++)
    if (((const uint8_t*)p)[k]) {
      dev().unclean++;
      return;
    }
}
void must_hold(const void* p, size_t bytes) {
  if (!inside(p, bytes)) dev().outside++;
}
template <typename T>
T arg(void** args, int k) {
  return *(T*)args[k];
}
uint64_t bricks_of(const VoxParams& P) {  // of the unit's segment
  const uint64_t end = morton3(P.pmax[0], P.pmax[1], P.pmax[2]) + 1;
  return (end - P.bstart + kBrickVox - 1) >> kBrickBits;
}
// the units' table segments, flags and cells: checked, then marked or cleared
enum { kTable = 1, kBytes = 2, kCells = 4, kPool = 8 };
void each(const VoxParams* units, uint32_t n, uint32_t* table, uint8_t* cflags, int what, int value) {
  for (uint32_t u = 0; u < n; u++) {
    const VoxParams& P = units[u];
    const uint64_t nb = bricks_of(P);
    if (what & kTable) {
      if (value < 0) must_be_zero(table + P.table_base, nb * 4);
      else if (nb * 4 <= kHuge && inside(table + P.table_base, nb * 4)) memset(table + P.table_base, value, nb * 4);
      if (P.wide) {
        uint8_t* f = cflags + P.table_base * kBrickWords;
        if (value < 0) must_be_zero(f, nb * kBrickWords);
        else if (nb * kBrickWords <= kHuge && inside(f, nb * kBrickWords)) memset(f, value, nb * kBrickWords);
      }
    }
    if (P.dense && (what & (P.wide ? kCells : kBytes))) {
      const size_t bytes = nb * kBrickVox * (P.wide ? 4 : 1);
      if (value < 0) must_be_zero(P.grid8, bytes);
      else if (bytes <= kHuge && inside(P.grid8, bytes)) memset(P.grid8, value, bytes);
    }
  }
}
struct Pass {
  const VoxParams* units;
  uint32_t n;
  ActArgs A;
} g_pass;
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) { return allocate(p, bytes); }
hipError_t hipFree(void* p) { return give_back(p); }
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) { return allocate(p, bytes); }
hipError_t hipHostFree(void* p) { return give_back(p); }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
  *f = *t = 256ull << 30;
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = dev().last;
  dev().last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 0;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t* s) {
  *s = (hipStream_t)1;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorUnknown; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipErrorUnknown; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  return hipErrorUnknown;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorUnknown; }
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = (hipEvent_t)1;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 0;
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t*, const void*) { return hipErrorInvalidValue; }
hipError_t hipMemGetAddressRange(hipDeviceptr_t*, size_t*, hipDeviceptr_t) { return hipErrorInvalidValue; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipSuccess; }
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*,
                           void*, void*, int*) {
  dev().names[f] = name;
}

hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t, hipStream_t) {
  Device& d = dev();
  look_for_stale();
  // HIP's limits: 2^32 - 1 threads along x, 1024 in a block
  if (!grid.x || (uint64_t)grid.x * block.x > 0xFFFFFFFFull || block.x > 1024) {
    d.bad_grid++;
    return d.last = hipErrorInvalidConfiguration;
  }
  const std::string& name = d.names[f];
  auto is = [&](const char* part) { return name.find(part) != std::string::npos; };
  if (is("k_fill_u32")) {
    uint32_t* p = arg<uint32_t*>(args, 0);
    const uint64_t n = arg<uint64_t>(args, 2);
    if (!inside(p, n * 4)) d.outside++;
    else if (n * 4 <= kHuge) std::fill(p, p + n, arg<uint32_t>(args, 1));
  } else if (is("k_fill_u64")) {
    uint64_t* p = arg<uint64_t*>(args, 0);
    const uint64_t n = arg<uint64_t>(args, 2);
    if (!inside(p, n * 8)) d.outside++;
    else if (n * 8 <= kHuge) std::fill(p, p + n, arg<uint64_t>(args, 1));
  } else if (is("k_gather_host")) {
    const GatherArgs g = arg<GatherArgs>(args, 0);
    for (int k = 0; k < g.n; k++) memcpy(g.dst[k], g.src[k], g.words[k] * 8);
    *arg<volatile uint32_t*>(args, 1) = arg<uint32_t>(args, 2);
  } else if (is("k_pass_begin")) {
    memset(arg<uint64_t*>(args, 0), 0, arg<uint64_t>(args, 1) * 8);
  } else if (is("k_vox_tile")) {
    g_pass = {arg<const VoxParams*>(args, 0), arg<uint32_t>(args, 1), arg<ActArgs>(args, 4)};
    const ActArgs& A = g_pass.A;
    d.marks++;
    if (is("TouchAction")) {
      each(g_pass.units, g_pass.n, A.table, A.cflags, kTable, -1);
      each(g_pass.units, g_pass.n, A.table, A.cflags, kTable, 1);
    } else if (is("MarkPool")) {
      must_be_zero(A.pool8, A.pool_cap * kBrickVox);
      if (inside(A.pool8, A.pool_cap * kBrickVox)) memset(A.pool8, 1, A.pool_cap * kBrickVox);
    } else if (is("WinnerAction")) {
      must_hold(A.pool, d.found * kBrickWords * 8);
      must_hold(A.wprefix, d.found * kBrickWords * 4);
      must_hold(A.winner, d.n_vox * 4);
    } else if (is("MarkDense") || is("MarkGather")) {
      d.dense++;
      each(g_pass.units, g_pass.n, A.table, A.cflags, kTable | kBytes | kCells, -1);
      each(g_pass.units, g_pass.n, A.table, A.cflags, kTable | kBytes | kCells, 1);
    }
  } else if (is("k_brick_count")) {
    ull* ctr = (ull*)g_pass.A.ctr;
    uint64_t all = 0;
    for (uint32_t u = 0; u < g_pass.n; u++) all += bricks_of(g_pass.units[u]);
    d.found = std::min(d.n_occ, all);
    ctr[kCtrNumOcc] = d.found;
    ctr[kCtrNumVox] = d.n_vox | (d.found << kNonEmptyShift);
    const uint64_t n = std::min(d.found, arg<uint64_t>(args, 2));
    must_hold(arg<ull*>(args, 8), n * kBrickWords * 8);  // the bricks' words and counts
    must_hold(arg<uint64_t*>(args, 9), n * 8);
    if (arg<uint64_t*>(args, 10)) must_hold(arg<uint64_t*>(args, 10), n * 8);
    if (arg<uint32_t*>(args, 12))  // a dense pass
      each(g_pass.units, g_pass.n, g_pass.A.table, g_pass.A.cflags, kTable | kBytes, 0);
    else if (inside(g_pass.A.pool8, g_pass.A.pool_cap * kBrickVox))
      memset(g_pass.A.pool8, 0, g_pass.A.pool_cap * kBrickVox);
  } else if (is("k_scan_single") && is("OccStoreDense")) {
    if (arg<uint64_t>(args, 2) > 1ull << kOccBits) d.outside++;  // (table indices of kOccBits)
  } else if (is("k_scan_single") && is("BrickOffStore")) {
    const BrickOffStore st = arg<BrickOffStore>(args, 1);
    if (st.host) {
      memcpy(st.host, st.ctr, kNumCounters * 8);
      *st.flag = (uint32_t)st.seq;
    }
  } else if (is("k_unit_voxels")) {  // the voxels dealt evenly to the units
    const uint32_t n = arg<uint32_t>(args, 4);
    for (uint32_t u = 0; u <= n; u++) arg<uint64_t*>(args, 6)[u] = d.n_vox * u / n;
  } else if (is("k_payload_bricks")) {
    each(g_pass.units, g_pass.n, nullptr, nullptr, kCells, 0);
  } else if (is("k_brick_emit")) {
    must_hold(arg<ull*>(args, 5), d.found * kBrickWords * 8);
    must_hold(arg<uint64_t*>(args, 6), d.found * 8);
    must_hold(arg<uint64_t*>(args, 10), d.found * kBrickWords * 8);
    if (arg<uint32_t*>(args, 8)) must_hold(arg<uint64_t*>(args, 7), d.n_vox * 8);
    if (arg<uint32_t*>(args, 8)) must_hold(arg<uint32_t*>(args, 8), d.found * kBrickWords * 4);
  } else if (is("k_brick_clear")) {
    each(g_pass.units, g_pass.n, g_pass.A.table, nullptr, kTable, 0);
  } else if (is("k_up_small") || is("k_up_scan") || is("k_build_init")) {
    // the build's bookkeeping: no flags, some nodes
    uint64_t* meta = *(uint64_t**)args[is("k_build_init") ? 0 : 1];
    memset(meta, 0, (2 * 64 + 8) * 8);
    meta[2 * 64 + 2] = 1000;
  }
  return hipSuccess;
}

// ---------------------------------------------------------------- what the test calls
// The next passes find n_occ bricks of n_vox voxels; the fail_at-th allocation from now on fails
// (-1: none does).
void state_found(uint64_t n_occ, uint64_t n_vox) {
  dev().n_occ = n_occ;
  dev().n_vox = n_vox;
}
void state_arm(long fail_at, uint64_t n_occ, uint64_t n_vox) {
  dev().allocs = 0;
  dev().fail_at = fail_at;
  state_found(n_occ, n_vox);
}
// out: allocations since arming, memory not zero when marked, accesses outside of allocations,
// grids that HIP refuses, mark kernels, those of dense passes, arguments in memory given back
void state_read(uint64_t out[7]) {
  Device& d = dev();
  out[0] = (uint64_t)d.allocs;
  out[1] = d.unclean;
  out[2] = d.outside;
  out[3] = d.bad_grid;
  out[4] = d.marks;
  out[5] = d.dense;
  out[6] = d.stale;
}
// A device-to-device copy of records.
int state_copy(uint64_t bytes) {
  Context c;
  const hipError_t e = copy_records(c, (void*)64, (const void*)128, bytes);
  if (c.hread) (void)hipHostFree(c.hread);
  return (int)e;
}
void state_clear() {
  Device& d = dev();
  d.unclean = d.outside = d.bad_grid = d.marks = d.dense = d.stale = 0;
  d.fail_at = -1;
  d.args.clear();
  t_launch_log = &d.args;
}
}
