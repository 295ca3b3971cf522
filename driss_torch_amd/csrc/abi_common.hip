// Status strings, device facts, tuning knobs and the workspace entry points of the C ABI.
#include <stdlib.h>
#include <string.h>
#include <strings.h>

#include <atomic>
#include <mutex>

#include "dt_device.hpp"
#include "dt_host.hpp"

namespace dt {

std::atomic<int> g_knob_values[] = {
#define DT_KNOB_VALUE(group, name, value) {value},
    DT_KNOBS(DT_KNOB_VALUE)
#undef DT_KNOB_VALUE
};

namespace {
// place of a key in the list of knobs, or -1
int knob_of(const char* key) {
  static const char* const keys[] = {
#define DT_KNOB_KEY(group, name, value) #group "." #name,
      DT_KNOBS(DT_KNOB_KEY)
#undef DT_KNOB_KEY
  };
  for (int i = 0; i < (int)Knob::count; ++i)
    if (strcmp(keys[i], key) == 0) return i;
  return -1;
}

// DRISS_TORCH_RESIDENT: "1", "on", "true", "yes" (any case) switch the one-kernel dynamic quantization on;
// anything else, or no variable, leaves it off.
bool resident_opt_in_from(const char* v) {
  if (!v) return false;
  for (const char* yes : {"1", "on", "true", "yes"})
    if (strcasecmp(v, yes) == 0) return true;
  return false;
}
struct KnobsFromEnvironment {
  KnobsFromEnvironment() {
    if (resident_opt_in_from(getenv("DRISS_TORCH_RESIDENT")))
      g_knob_values[(int)Knob::dynamic_resident].store(1, std::memory_order_relaxed);
  }
} g_knobs_from_environment;  // when the library is loaded; the values above are there before (constant-initialised)

#ifdef DT_PHASE_LOG
std::atomic<uint64_t*> g_phase_log{nullptr};
std::atomic<size_t> g_phase_log_bytes{0};
std::atomic<int> g_phase_log_device{-1};
#endif

constexpr int kMaxDevices = 16;
DeviceFacts g_facts[kMaxDevices];
std::once_flag g_facts_once[kMaxDevices];
}  // namespace

#ifdef DT_PHASE_LOG
uint64_t* phase_log(size_t need_bytes) {
  uint64_t* p = g_phase_log.load(std::memory_order_relaxed);
  if (!p || g_phase_log_bytes.load(std::memory_order_relaxed) < need_bytes) return nullptr;
  int dev = -1;
  (void)hipGetDevice(&dev);
  return dev == g_phase_log_device.load(std::memory_order_relaxed) ? p : nullptr;  // the buffer's own device only
}
#endif

const DeviceFacts& device_facts() {
  int dev = 0;
  (void)hipGetDevice(&dev);
  if (dev < 0 || dev >= kMaxDevices) dev = 0;
  std::call_once(g_facts_once[dev], [dev] {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
    g_facts[dev].cu_count = cus;
  });
  return g_facts[dev];
}

__global__ void zero_words_kernel(uint32_t* p, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

}  // namespace dt

extern "C" {

const char* dt_status_string(int status) {
  switch (status) {
    case DT_OK: return "ok";
    case DT_ERR_INVALID_DTYPE: return "unsupported dtype";
    case DT_ERR_INVALID_SHAPE: return "invalid shape";
    case DT_ERR_NULL_POINTER: return "null pointer";
    case DT_ERR_MISALIGNED: return "misaligned pointer";
    case DT_ERR_WORKSPACE: return "workspace missing or too small";
    case DT_ERR_INVALID_MODE: return "invalid mode";
    case DT_ERR_LAUNCH: return "kernel launch failed";
    case DT_ERR_EMPTY: return "reduction over zero elements";
    case DT_ERR_RESIDENT_GAVE_UP:
      return "an earlier dynamic quantization on this device gave up waiting for the whole chip and wrote NaN "
             "(is another process using the GPU?); the one-kernel path is now off for this process";
    case DT_ERR_TOO_LARGE: return "more elements than the no-allocation entry point takes (DT_NOALLOC_MAX_NUMEL)";
    default: return "unknown status";
  }
}

int dt_abi_version(void) { return 1; }

size_t dt_workspace_bytes(void) { return dt::kWsBytes; }

int dt_workspace_init(void* workspace, size_t workspace_bytes, dt_stream_t stream) {
  if (!workspace) return DT_ERR_NULL_POINTER;
  if (workspace_bytes < dt::kWsBytes) return DT_ERR_WORKSPACE;
  if (!dt::aligned(workspace, 256)) return DT_ERR_MISALIGNED;
  // a fill kernel rather than hipMemsetAsync, so the call is safe under graph capture
  dt::launcher(dt::zero_words_kernel, dt::kWsBytes / 4 / 256, 256, 0, dt::as_hip(stream))(static_cast<uint32_t*>(workspace), dt::kWsBytes / 4);
  return dt::launch_status();
}

#ifdef DT_PHASE_LOG
int dt_set_phase_log(void* device_buffer, size_t bytes) {
  if (device_buffer && !dt::aligned(device_buffer, 8)) return DT_ERR_MISALIGNED;
  int dev = -1;
  (void)hipGetDevice(&dev);
  dt::g_phase_log.store(nullptr, std::memory_order_relaxed);
  dt::g_phase_log_bytes.store(device_buffer ? bytes : 0, std::memory_order_relaxed);
  dt::g_phase_log_device.store(device_buffer ? dev : -1, std::memory_order_relaxed);
  dt::g_phase_log.store(static_cast<uint64_t*>(device_buffer), std::memory_order_relaxed);
  return DT_OK;
}
#endif

int dt_set_tuning(const char* key, int value) {
  if (!key) return DT_ERR_NULL_POINTER;
  const int i = dt::knob_of(key);
  if (i < 0) return DT_ERR_INVALID_MODE;
  dt::g_knob_values[i].store(value, std::memory_order_relaxed);
  return DT_OK;
}

int dt_get_tuning(const char* key, int* value) {
  if (!key || !value) return DT_ERR_NULL_POINTER;
  const int i = dt::knob_of(key);
  if (i < 0) return DT_ERR_INVALID_MODE;
  *value = dt::g_knob_values[i].load(std::memory_order_relaxed);
  return DT_OK;
}

}  // extern "C"
