// A host stand-in for the HIP runtime and the kernel launchers, linked with
// the library's context.cpp so that its buffer management runs on the CPU.
// Device memory is host memory.  Every allocation is recorded, freed blocks
// are never handed out again, and no kernel runs: each launch instead checks
// that what its kernel would reach lies inside live allocations of at least
// the size that it would read or write.  What does not is kept as a line of
// text for host_device_faults().
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

#include "../mepgl_amd/csrc/common.hpp"
#include "../mepgl_amd/csrc/field_io.hpp"
#include "../mepgl_amd/csrc/gauge_local.hpp"
#include "../mepgl_amd/csrc/kernels.hpp"

namespace {

std::map<const char*, size_t> live;
std::string faults;

void* take(size_t bytes) {
  void* p = std::calloc(bytes ? bytes : 1, 1);
  live[(const char*)p] = bytes;
  return p;
}

hipError_t give_back(void* p) {
  if (p && !live.erase((const char*)p)) faults += "a block freed twice\n";
  return hipSuccess;  // the memory itself stays, so that its address never comes again
}

bool inside(const void* p, size_t bytes) {
  auto it = live.upper_bound((const char*)p);
  if (!p || it == live.begin()) return false;
  --it;
  return (const char*)p + bytes <= it->first + it->second;
}

void need(const std::string& what, const void* p, size_t bytes) {
  if (!inside(p, bytes))
    faults += what + ": " + std::to_string(bytes) + " bytes not in a live allocation\n";
}

// Everything that a kernel can reach through a string's descriptor.
void check_string(const mepgl::DevString& s, const std::string& where, bool fp32) {
  using namespace mepgl;
  const size_t elem = fp32 ? 4 : 8, F = (size_t)s.F, tiles = F * s.tiles_x * s.tiles_y;
  const size_t fields = F * s.image_stride, plane = (size_t)s.N * s.pitch;
  if (s.tiles_y != (s.N + s.seg_rows - 1) / s.seg_rows) faults += where + ": tiles_y\n";
  for (int b = 0; b < 2; ++b) {
    need(where + " fields", s.x[b], fields * elem);
    need(where + " directions", s.d[b], fields * elem);
    need(where + " gradients", s.g[b], fields * elem);
  }
  need(where + " partials of G", s.part_g, tiles * kPartG * 8);
  need(where + " partials of P", s.part_p, tiles * kPartP * 8);
  need(where + " partials of the arclength", s.part_a, tiles * kPartA * 8);
  need(where + " spline system", s.cubic, F * kCubicCoefs * 8);
  need(where + " plan weights", s.plan_w, F * 8);
  need(where + " plan nodes", s.plan_k, F * sizeof(int));
  need(where + " spline plan weights", s.cplan_w, F * 8);
  need(where + " spline plan nodes", s.cplan_k, F * sizeof(int));
  need(where + " neighbour map", s.nn, plane * sizeof(uint16_t));
  if (s.gs) need(where + " scratch gradient", s.gs, fields * elem);
  if (s.cubic_rhs) need(where + " spline right-hand sides", s.cubic_rhs, fields * 8);
  const DevParam* params[] = {&s.a[0], &s.b[0], &s.mxx[0], &s.myy[0], &s.a[1],
                              &s.b[1], &s.mxx[1], &s.myy[1], &s.h};
  bool planes = false;
  for (auto* p : params) {
    planes = planes || p->p;
    if (p->p) need(where + " parameter plane", p->p, plane * 8);
  }
  if (planes)
    need(where + " derived parameter planes", s.prm,
         (size_t)(kParamPlanes * s.nc + 1) * s.N * s.plane_stride * elem);
}

void check_items(const char* launch, const mepgl::DevString* strings, const mepgl::WorkItem* items,
                 int nitems, bool fp32) {
  const std::string where = std::string(launch) + ": string ";
  need(std::string(launch) + " items", items, sizeof(mepgl::WorkItem) * nitems);
  int last = -1;
  for (int k = 0; k < nitems && inside(items + k, sizeof *items); ++k) {
    const mepgl::WorkItem& it = items[k];
    const mepgl::DevString& s = strings[it.string];
    const std::string at = where + std::to_string(it.string);
    if (it.string != last) check_string(s, at, fp32);
    last = it.string;
    if (it.image < 0 || it.image >= s.F || it.tile < 0 || it.tile >= s.tiles_x * s.tiles_y)
      faults += at + ": an item outside the string\n";
  }
}

}  // namespace

extern "C" {

const char* host_device_faults() { return faults.c_str(); }
void host_device_clear() { faults.clear(); }

// Bytes in live allocations.
long long host_device_bytes() {
  long long n = 0;
  for (auto& a : live) n += (long long)a.second;
  return n;
}

hipError_t hipMalloc(void** p, size_t n) { return *p = take(n), hipSuccess; }
hipError_t hipFree(void* p) { return give_back(p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return *p = take(n), hipSuccess; }
hipError_t hipHostFree(void* p) { return give_back(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) {
  if (k != hipMemcpyDeviceToHost) need("copy to the device", d, n);
  if (k != hipMemcpyHostToDevice) need("copy from the device", s, n);
  return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) {
  need("fill", p, n);
  return std::memset(p, v, n), hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "host stand-in"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = (hipStream_t)take(1), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return give_back(s); }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  return hipErrorNotSupported;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = (hipEvent_t)take(1), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return give_back(e); }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
// Every timing is equal: the tuner keeps the first candidate of each class,
// the height that its first string has.
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1, hipSuccess; }

}  // extern "C"

namespace mepgl {

hipError_t launch_step(const StepArgs& a, int, bool fp32, hipStream_t) {
  check_items("step", a.strings, a.items, a.nitems, fp32);
  return hipSuccess;
}
hipError_t launch_aux(const AuxArgs& a, int, int, bool fp32, hipStream_t) {
  check_items("auxiliary pass", a.strings, a.items, a.nitems, fp32);
  return hipSuccess;
}
hipError_t launch_finish(const FinishArgs& f, int, bool, hipStream_t) {
  need("finishing launch scalars", f.sc, sizeof(ImageScalars) * f.nimages);
  need("finishing launch results", f.out, sizeof(double) * f.nimages);
  return hipSuccess;
}
hipError_t launch_glocal(const AuxArgs& a, int, bool fp32, hipStream_t) {
  check_items("local alignment", a.strings, a.items, a.nitems, fp32);
  return hipSuccess;
}
// The operand that all images share is the N x N cosine matrix; the
// eigenvalues follow it.
hipError_t launch_dct_gemm(const GemmArgs& g, int, hipStream_t) {
  const size_t n = (size_t)g.n;
  need("cosine matrix", g.abatch ? g.B : g.A, n * n * 8);
  need("product", g.O, n * 8);
  if (g.lam) need("eigenvalues", g.lam, n * 8);
  return hipSuccess;
}
hipError_t launch_glocal_prefix(double*, int, int, long long, long long, hipStream_t) { return hipSuccess; }
hipError_t launch_derive_params(const DevString& s, bool fp32, hipStream_t) {
  need("derived parameter planes", s.prm,
       (size_t)(kParamPlanes * s.nc + 1) * s.N * s.plane_stride * (fp32 ? 4 : 8));
  return hipSuccess;
}
// Every site has all its bonds.
hipError_t launch_nn_map(const int*, const int*, int N, int pitch, uint16_t* nn, hipStream_t) {
  std::memset(nn, 0xff, (size_t)N * pitch * sizeof(uint16_t));
  return hipSuccess;
}
hipError_t launch_fill(void* p, long long n, bool fp32, double, hipStream_t) {
  need("fill", p, (size_t)n * (fp32 ? 4 : 8));
  return hipSuccess;
}

void FieldIo::release() {}
hipError_t download_fields(FieldIo&, const DevString& d, const void* dev, bool fp32,
                           const HostField* f, int nf, const hipStream_t*, int, int) {
  need("download", dev, (size_t)d.F * d.image_stride * (fp32 ? 4 : 8));
  for (int k = 0; k < nf; ++k)
    std::memset(f[k].host, 0, sizeof(double) * d.F * d.N * d.N * f[k].count);
  return hipSuccess;
}
hipError_t upload_fields(FieldIo&, const DevString& d, void* const* dev, int ndev, bool fp32,
                         const HostField*, int, const hipStream_t*, int, int) {
  for (int k = 0; k < ndev; ++k) need("upload", dev[k], (size_t)d.F * d.image_stride * (fp32 ? 4 : 8));
  return hipSuccess;
}
bool images_equal(const double* a, int F, size_t image) {
  for (int n = 1; n < F; ++n)
    if (std::memcmp(a, a + (size_t)n * image, image * sizeof(double)) != 0) return false;
  return true;
}

}  // namespace mepgl
