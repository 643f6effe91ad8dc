// The C-ABI layer (lbf_api.cpp) over a HIP runtime and kernels that do nothing:
// its host logic -- tiles, allocation failures, what each launch is given -- runs
// without a GPU.  Device memory is host memory; hipMalloc fails from the
// allocation on that stub_fail_after() names.
#include "../../lbfast_amd/csrc/lbf_api.cpp"
#include "../../lbfast_amd/csrc/lbf_physics.h"
#include <cstdlib>

static long g_left = -1;  // allocations until hipMalloc fails; -1: never
static lbf::FusedArgs g_fused;
static lbf::StageArgs g_wetting;
static int g_prep_tz;

extern "C" {
void stub_fail_after(long n) { g_left = n; }
void stub_fused_tile(int* ty, int* tz) { *ty = g_fused.ty; *tz = g_fused.tz; }
int stub_prep_chunk() { return g_prep_tz; }
// of the last wetting update: the list's length, and the haloed isfluid's sum and
// number of wall words
void stub_wetting(long* out) {
  const size_t n = lbf::halo_nodes(g_wetting.dp);
  out[0] = g_wetting.nwet;
  out[1] = out[2] = 0;
  for (size_t i = 0; i < n; ++i) {
    out[1] += g_wetting.isfh[i];
    out[2] += g_wetting.words[i] != 0;
  }
}

hipError_t hipMalloc(void** p, size_t n) {
  *p = g_left == 0 ? nullptr : calloc(1, n);
  if (g_left > 0) --g_left;
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "stub"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t* s) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) { return hipErrorNotSupported; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = nullptr; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = nullptr; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }
}

namespace lbf {
bool default_scales(const DevParams&) { return true; }
int fused_tile_count(const FusedArgs&) { return 1; }
int prep_tile_count(const StageArgs& a, int tz) {
  return ((a.dp.nx + 63) / 64) * ((a.dp.ny + 11) / 12) * ((a.dp.nz + tz - 1) / tz);
}
hipError_t launch_fused(const FusedArgs& a, int, bool, hipStream_t) { g_fused = a; return hipSuccess; }
hipError_t launch_stage(int stage, const StageArgs& a, int, hipStream_t) {
  if (stage == LBF_STAGE_PHI_INT_BOUNDARY) g_wetting = a;
  return hipSuccess;
}
// one list entry for each solid node of the haloed array
hipError_t launch_wet_list(const int8_t* isfh, void*, uint32_t* count, const DevParams& dp, int, hipStream_t) {
  for (size_t i = 0; i < halo_nodes(dp); ++i) *count += isfh[i] == 0;
  return hipSuccess;
}
hipError_t launch_node_words(const int8_t* isfh, uint32_t* words, const DevParams& dp, hipStream_t) {
  for (size_t i = 0; i < halo_nodes(dp); ++i) words[i] = isfh[i] == 0;
  return hipSuccess;
}
hipError_t launch_fill_zero(void* p, size_t n, hipStream_t) { if (n < 64) memset(p, 0, n); return hipSuccess; }
hipError_t launch_copy(void* d, const void* s, size_t n, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t launch_fused_batch(const FusedBatchEntry*, int, int, int, int, bool, bool, bool, int, hipStream_t) { return hipSuccess; }
hipError_t launch_phase_prep(const StageArgs&, int, int tz, hipStream_t) { g_prep_tz = tz; return hipSuccess; }
hipError_t launch_phase_prep_batch(const PrepBatchEntry*, int, int, int, hipStream_t) { return hipSuccess; }
hipError_t launch_encode_moments(void*, const float*, const DevParams&, int, hipStream_t) { return hipSuccess; }
hipError_t launch_decode_field(const void*, int, void*, int, const DevParams&, int, hipStream_t) { return hipSuccess; }
hipError_t launch_convert_in(const void*, int, void*, int, FieldLay, const DevParams&, float, hipStream_t) { return hipSuccess; }
hipError_t launch_convert_out(const void*, int, FieldLay, void*, int, const DevParams&, float, hipStream_t) { return hipSuccess; }
hipError_t launch_set_copy(void*, FieldLay, const void*, FieldLay, int, int, const DevParams&, hipStream_t) { return hipSuccess; }
hipError_t launch_reduce(const void*, const void*, const int8_t*, const DevParams&, int, double*, int, double*, hipStream_t) { return hipSuccess; }
hipError_t launch_reduce_scratch(const void*, const void*, const int8_t*, const DevParams&, int, double*, hipStream_t) { return hipSuccess; }
hipError_t reduce_scratch_ptr(int, double**) { return hipErrorNotSupported; }
hipError_t launch_phi_lagrange(const StageArgs&, int, double*, int, double*, bool, hipStream_t) { return hipSuccess; }
hipError_t launch_tick(uint32_t*, int, hipStream_t) { return hipSuccess; }
}  // namespace lbf
