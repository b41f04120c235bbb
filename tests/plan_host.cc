// plan_host.cc -- the routes of u15h_api.cc on the host, for test_plan.py.
//
// The API's own source, compiled with the HIP calls and the kernel launchers
// it makes replaced by the ones below, which print what they are asked for.
// Reads one call per line from stdin:
//   linear M K N | pack bits group M K N | mot M_und M_gen K N |
//   swiglu M_und M_gen K I | i8 M_und M_gen K N |
//   attn hq hkv tq tk d q_offset mode
// ("captured" before it: on a capturing stream), each on a context of its own, and prints a line per call: its launches (and
// device allocations after u15h_create, "malloc relaxed" where the thread's
// capture mode lets a capturing stream's caller allocate), separated by
// " ; ", then the status.
// A batch that the kernels would refuse, or whose partial sums do not fit the
// scratch, is answered as they answer it: with hipErrorInvalidValue.  The
// first argument is the number of CUs.
#include "u15h_api.cc"

#include <iostream>
#include <sstream>

namespace {

int g_cus = 256;
bool g_created = false;
hipStreamCaptureMode g_mode = hipStreamCaptureModeGlobal;
bool g_capturing = false;
std::string g_out;

void
emit(const std::string& s)
{
  g_out += s + " ; ";
}

// Non-null and aligned; nothing on the host reads through it.
template <class T>
T*
fake(uintptr_t at = 4096)
{
  return reinterpret_cast<T*>(at);
}

const char*
epi_name(u15h::Epi e)
{
  const char* const names[] = {"bf16", "i32", "i8", "swiglu"};
  return names[(int)e];
}

hipError_t
tiled(const char* what, const u15h::GemmBatch& b, u15h::Epi epi)
{
  const bool mid = b.bn == u15h::kMidBN && (b.bm == 128 || b.bm == 192 || b.bm == 256);
  if (!mid && (b.bm != u15h::kBM || b.bn != u15h::kBN)) { return hipErrorInvalidValue; }
  int tiles = 0;
  for (int i = 0; i < b.nprob; ++i) {
    const u15h::GemmProblem& p = b.p[i];
    const int cols = u15h::tile_cols(epi, b.bn);
    if (p.tile_begin != tiles || p.tiles_m != (p.rows + b.bm - 1) / b.bm ||
        p.tiles_n != (p.n + cols - 1) / cols) {
      return hipErrorInvalidValue;
    }
    tiles += p.tiles_m * p.tiles_n;
  }
  const size_t cap = (size_t)g_cus * u15h::kBM * u15h::kBN * 4;
  if (tiles != b.total_tiles || (b.split > 1 && (b.ws == nullptr || split_ws_bytes(b) > cap))) {
    return hipErrorInvalidValue;
  }
  std::ostringstream s;
  s << what << " " << epi_name(epi) << " " << b.bm << "x" << b.bn << " tiles=" << b.total_tiles
    << " tail=" << b.total_tiles - b.split_begin << " shares=" << b.split;
  emit(s.str());
  return hipSuccess;
}

hipError_t
skinny(const u15h::SkinnyBatch& b, const char* type)
{
  const size_t cap = (size_t)g_cus * u15h::kBM * u15h::kBN * 4;
  if (b.max_rows > u15h::kSkinnyMaxRows || b.kbytes % 128 != 0 ||
      (b.split > 1 && (b.ws == nullptr || u15h::skinny_ws_floats(b) * 4 > cap))) {
    return hipErrorInvalidValue;
  }
  std::ostringstream s;
  s << "skinny " << type << " rows=" << b.max_rows << " cols=" << b.cols << " waves=" << b.waves
    << " shares=" << b.split;
  emit(s.str());
  return hipSuccess;
}

}  // namespace

namespace u15h {

hipError_t
launch_gemm_bf16(const GemmBatch& b, Epi epi, const GemmShape&, hipStream_t, const GemmEvents&)
{
  return tiled("tiled", b, epi);
}
hipError_t
launch_gemm_i8(const GemmBatch& b, Epi epi, const GemmShape&, hipStream_t, const GemmEvents&)
{
  return tiled("tiled", b, epi);
}
hipError_t
launch_gemm_pack(const GemmBatch& b, int, int, const GemmShape&, hipStream_t, const GemmEvents&)
{
  return b.bn != kMidBN || b.kbytes % 128 != 0 ? hipErrorInvalidValue
                                               : tiled("pack", b, Epi::kBf16);
}
hipError_t
launch_skinny_bf16(const SkinnyBatch& b, hipStream_t, const GemmEvents&)
{
  return skinny(b, b.qbits != 0 ? "pack" : b.swiglu ? "swiglu" : "bf16");
}
hipError_t
launch_skinny_i8(const SkinnyBatch& b, Epi epi, hipStream_t, const GemmEvents&)
{
  return skinny(b, epi_name(epi));
}
hipError_t
launch_dequant_affine(const uint32_t*, const uint16_t*, const uint16_t*, int, int, int, int,
                      uint16_t*, hipStream_t)
{
  emit("expand");
  return hipSuccess;
}
hipError_t
launch_attention(const AttnArgs& a, hipStream_t)
{
  if (a.shares > 1 && (a.ws == nullptr || attn_split_ws_bytes(a) > kAttnWsBytes)) {
    return hipErrorInvalidValue;
  }
  emit("attention shares=" + std::to_string(a.shares));
  return hipSuccess;
}
hipError_t
launch_quant_rows_i8(const uint16_t*, int, int, int8_t*, float*, hipStream_t, hipEvent_t,
                     hipEvent_t)
{
  emit("quant");
  return hipSuccess;
}
bool kernels_loadable() { return true; }
hipError_t
noalloc_scratch(int, void** out)
{
  *out = fake<void>();
  return hipSuccess;
}
// not called here
hipError_t launch_swiglu(const uint16_t*, const uint16_t*, uint16_t*, int64_t, hipStream_t)
{ return hipErrorUnknown; }
hipError_t launch_add_bf16(uint16_t*, const uint16_t*, int64_t, hipStream_t)
{ return hipErrorUnknown; }
hipError_t launch_bias_add(uint16_t*, const uint16_t*, int, int, hipStream_t)
{ return hipErrorUnknown; }
hipError_t launch_rms_norm(uint16_t*, const uint16_t*, const uint16_t*, const uint16_t*, int, int,
                           int, float, uint16_t*, int8_t*, float*, hipStream_t)
{ return hipErrorUnknown; }
hipError_t launch_f16_to_bf16(const uint16_t*, int64_t, uint16_t*, hipStream_t)
{ return hipErrorUnknown; }
hipError_t launch_f32_to_bf16(const float*, int64_t, uint16_t*, hipStream_t)
{ return hipErrorUnknown; }
hipError_t launch_gather_rows(const uint16_t*, const int32_t*, int, int, uint16_t*, bool,
                              hipStream_t)
{ return hipErrorUnknown; }
hipError_t launch_swiglu_quant(const uint16_t*, const uint16_t*, int, int, uint16_t*, int8_t*,
                               float*, hipStream_t)
{ return hipErrorUnknown; }
hipError_t launch_transpose_rows(const uint16_t*, uint16_t*, int, int, int, long long, long long,
                                 long long, long long, hipStream_t)
{ return hipErrorUnknown; }
hipError_t launch_split_norm_rope(uint16_t*, const uint16_t*, const uint16_t*, const float*,
                                  const float*, int, int, int, int, int, float, bool, bool,
                                  hipStream_t)
{ return hipErrorUnknown; }
hipError_t launch_attention_prologue(const PrologueArgs&, hipStream_t, int)
{ return hipErrorUnknown; }

}  // namespace u15h

extern "C" {

hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipFree(void*) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t
hipGetDeviceProperties(hipDeviceProp_t* p, int)    // a macro for the versioned name
{
  std::memset(p, 0, sizeof *p);
  std::strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = g_cus;
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "refused"; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t
hipMalloc(void** p, size_t)
{
  if (g_created) {
    emit(g_mode == hipStreamCaptureModeRelaxed ? "malloc relaxed" : "malloc");
  }
  *p = fake<void>();
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t
hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* status)
{
  *status = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t
hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* mode)
{
  std::swap(*mode, g_mode);
  return hipSuccess;
}

}  // extern "C"

int
main(int argc, char** argv)
{
  if (argc > 1) { g_cus = std::atoi(argv[1]); }
  std::string line;
  while (std::getline(std::cin, line)) {
    std::istringstream in(line);
    std::string call;
    in >> call;
    g_capturing = call == "captured";
    if (g_capturing) { in >> call; }
    int v[7] = {};
    for (int& x : v) { in >> x; }
    g_out.clear();
    g_created = false;
    u15h_ctx* ctx = nullptr;
    if (u15h_create(0, &ctx) != U15H_OK) { return 1; }
    g_created = true;
    u15h_bf16* const t = fake<u15h_bf16>();
    u15h_status st = U15H_EINVAL;
    if (call == "linear") {
      st = u15h_linear(ctx, nullptr, t, t, nullptr, t, v[0], v[1], v[2]);
    } else if (call == "pack") {
      const u15h_qweight w = {fake<uint32_t>(), t, t, v[0], v[1]};
      st = u15h_linear_q(ctx, nullptr, t, &w, nullptr, t, v[2], v[3], v[4]);
    } else if (call == "mot") {
      const u15h_mot_proj p = {t, t, nullptr, nullptr, t, v[3]};
      st = u15h_mot_linear(ctx, nullptr, t, v[0], v[1], v[2], &p, 1);
    } else if (call == "swiglu") {
      st = u15h_mot_gate_up_swiglu(ctx, nullptr, t, v[0], v[1], v[2], t, t, t, t, t, v[3]);
    } else if (call == "i8") {
      u15h_mot_proj_i8 p;
      std::memset(&p, 0, sizeof p);
      p.wq_und = p.wq_gen = fake<int8_t>();
      p.sw_und = p.sw_gen = fake<float>();
      p.y = t;
      p.N = v[3];
      st = u15h_mot_gemm_i8(ctx, nullptr, fake<int8_t>(), fake<float>(), v[0], v[1], v[2], &p, 1);
    } else if (call == "attn") {
      st = u15h_attention_token_major(ctx, nullptr, t, t, t, t, fake<int32_t>(), v[0], v[1], v[2],
                                      v[3], v[4], v[3], v[5], v[6]);
    }
    std::cout << g_out << u15h_status_str(st) << "\n";
    u15h_destroy(ctx);
  }
  return 0;
}
