// What the library's host code launches and where it points the kernels, on
// the CPU: this program stands in for the HIP runtime (its definitions come
// before libamdhip64's), records every launch with a copy of the kernel's
// parameters and runs none of them. Device pointers are addresses nobody reads.
//
// Prints "ok <case>" per case; exits nonzero at the first failure.

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "dn_common.hpp"
#include "mfma_scan.hpp"

namespace {

struct Launch {
  std::string kernel;
  const void* params;  // valid until the next launch
  int threads;
};

std::map<const void*, std::string>& kernels() {
  static auto* m = new std::map<const void*, std::string>();  // filled before main
  return *m;
}

int device = 0;  // current device: how many CUs it has
const int kCus[] = {256, 128, 64, 32};
int blocks_per_cu = 0;  // what the occupancy query answers
void (*on_launch)(const Launch&) = nullptr;
int launches = 0, failing = 0;  // the launch whose check reports an error, from 1; 0: none
// Waits of the second stream for the caller's, and of the caller's for it.
int forks = 0, joins = 0;
const hipStream_t kSide = reinterpret_cast<hipStream_t>(uintptr_t(1) << 12);

void fail(const std::string& what) {
  std::fprintf(stderr, "FAIL %s\n", what.c_str());
  std::exit(1);
}

hipError_t record(const void* f, dim3 block, void** args) {
  const auto it = kernels().find(f);
  if (it == kernels().end()) fail("launch of an unregistered kernel");
  if (on_launch) on_launch({it->second, args[0], int(block.x)});
  ++launches;
  return hipSuccess;
}

}  // namespace

extern "C" {
void** __hipRegisterFatBinary(const void*) {
  static void* handle = nullptr;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, uint3*,
                           uint3*, dim3*, dim3*, int*) {
  kernels()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
static dim3 pushed;  // the block of the launch under way
hipError_t __hipPushCallConfiguration(dim3, dim3 block, size_t, hipStream_t) {
  pushed = block;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3*, dim3* block, size_t*, hipStream_t*) {
  *block = pushed;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3 block, void** args, size_t, hipStream_t) {
  return record(f, block, args);
}
hipError_t hipLaunchCooperativeKernel(const void* f, dim3, dim3 block, void** args, unsigned,
                                      hipStream_t) {
  return record(f, block, args);
}
hipError_t hipGetLastError() {
  return failing && launches == failing ? hipErrorLaunchFailure : hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = kSide;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t*, unsigned) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t, unsigned) {
  ++(s == kSide ? forks : joins);
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = device;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int d) {
  *v = kCus[d];
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = blocks_per_cu;
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t) {
  *p = reinterpret_cast<void*>(uintptr_t(1) << 20);
  return hipSuccess;
}
hipError_t hipMemset(void*, int, size_t) { return hipSuccess; }
}

namespace {

char* const kWorkspace = reinterpret_cast<char*>(uintptr_t(1) << 44);
const void* const kTensor = reinterpret_cast<const void*>(uintptr_t(1) << 30);

dn_chunk_fwd_args forward(int B, int S, int H, int K, int V, bool channel) {
  dn_chunk_fwd_args a{};
  a.batch = B, a.sequence = S, a.nheads = H, a.head_k_dim = K, a.head_v_dim = V;
  a.erase_width = channel ? K : 1, a.write_width = channel ? V : 1;
  a.decay_width = channel ? K : 1;
  a.has_gate = 1, a.chunk_len = 64, a.scale = std::nan("");
  a.qkv_dtype = a.y_dtype = DN_BF16;
  a.q = a.k = a.v = kTensor;
  a.erase = a.write = a.g = a.state_in = static_cast<const float*>(kTensor);
  a.y = const_cast<void*>(kTensor);
  a.state_out = static_cast<float*>(const_cast<void*>(kTensor));
  a.workspace = kWorkspace;
  return a;
}

// The end of the segmented scan's buffers, as its carry kernel is given them.
struct Segments {
  int parts = 0;
  const char* end = nullptr;
} segments;

void see_segments(const Launch& l) {
  if (l.kernel.find("seg_carry_kernel") == std::string::npos) return;
  const auto& p = *static_cast<const dn::MfmaParams*>(l.params);
  const int K = l.kernel.find("Li128E") != std::string::npos ? 128 : 64;
  segments.parts = p.seg_p;
  segments.end = reinterpret_cast<const char*>(p.seg_start + size_t(p.B) * p.seg_p * p.H * K * p.V);
}

// dn_chunk_fwd_out_norm with the norm in the scan, on devices where its
// cooperative launch never fits: the plain forward runs in its workspace.
void out_norm_fallback() {
  on_launch = see_segments;
  blocks_per_cu = 0;
  int cut = 0;
  for (device = 0; device < 4; ++device)
    for (int K : {64, 128})
      for (int V = 64; V <= 1024; V += 64)
        for (int chunks : {32, 64, 100, 256})
          for (int heads : {1, 2, 3, 5})
            for (bool channel : {false, true}) {
              dn_chunk_fwd_out_norm_args a{};
              a.fwd = forward(1, 64 * chunks, heads, K, V, channel);
              a.weight = static_cast<const float*>(kTensor);
              a.eps = 1e-5;
              a.in_scan = 1;
              a.fwd.workspace_bytes = dn_chunk_fwd_out_norm_workspace_bytes(&a);
              segments = {};
              if (dn_chunk_fwd_out_norm(&a, nullptr) != DN_OK) fail(dn_last_error());
              cut += segments.parts > 1;
              if (segments.end > kWorkspace + a.fwd.workspace_bytes)
                fail("out norm fallback: " + std::to_string(segments.parts) + " segments of K " +
                     std::to_string(K) + " V " + std::to_string(V) + " chunks " +
                     std::to_string(chunks) + " heads " + std::to_string(heads) + " end " +
                     std::to_string(segments.end - kWorkspace - a.fwd.workspace_bytes) +
                     " bytes past the workspace");
            }
  device = 0;
  if (!cut) fail("out norm fallback: no call was segmented");
  std::printf("ok out_norm_fallback (%d segmented calls)\n", cut);
}

// A workspace of the size that fewer segments, or none, took serves the call,
// which keeps to it; a smaller one is refused.
void smaller_workspaces() {
  on_launch = see_segments;
  const struct {
    int S, K, V;
    size_t bytes;
  } cases[] = {{4096, 64, 128, 1589760}, {4096, 128, 576, 1591552}, {8192, 128, 192, 3179264},
               {16384, 64, 576, 6359296}, {2048, 64, 64, 794880},
               {8192, 128, 256, 3179520}};
  for (const auto& c : cases) {
    dn_chunk_fwd_args a = forward(1, c.S, 1, c.K, c.V, false);
    if (dn_chunk_fwd_workspace_bytes(&a) <= c.bytes) fail("smaller workspace: not smaller");
    for (size_t more : {size_t(0), size_t(1) << 19, size_t(1) << 26}) {
      a.workspace_bytes = c.bytes + more;
      segments = {};
      if (dn_chunk_fwd(&a, nullptr) != DN_OK) fail(dn_last_error());
      if (segments.end > kWorkspace + a.workspace_bytes) fail("smaller workspace: left");
      if (more > dn_chunk_fwd_workspace_bytes(&a) && segments.parts < 2)
        fail("smaller workspace: a large one is not cut");
    }
    a.workspace_bytes = c.bytes - 1;
    if (dn_chunk_fwd(&a, nullptr) != DN_ERR_WORKSPACE) fail("smaller workspace: accepted");
  }
  std::printf("ok smaller_workspaces\n");
}

// Which kernels walk the segments: teams where a round of the device holds
// them, 8-wave workgroups where it does not, or the sequence whole.
void segment_kernels() {
  static int teams, lone, carries;
  on_launch = [](const Launch& l) {
    teams += l.kernel.find("team_scan_kernel") != std::string::npos;
    lone += l.kernel.find("mfma_scan_kernel") != std::string::npos;
    carries += l.kernel.find("seg_carry_kernel") != std::string::npos;
  };
  const struct {
    int S, H, V;
    bool channel;
    int teams, lone, carries;
  } cases[] = {{12288, 4, 256, false, 2, 0, 1}, {16384, 8, 256, false, 0, 2, 1},
               {16384, 8, 256, true, 0, 2, 1},  {16384, 4, 256, true, 2, 0, 1},
               {16384, 16, 128, false, 0, 2, 1}, {16384, 6, 192, false, 2, 0, 1},
               {16352, 8, 256, false, 1, 0, 0}, {2048, 16, 256, false, 1, 0, 0}};
  for (const auto& c : cases) {
    dn_chunk_fwd_args a = forward(1, c.S, c.H, 128, c.V, c.channel);
    a.workspace_bytes = dn_chunk_fwd_workspace_bytes(&a);
    teams = lone = carries = 0;
    if (dn_chunk_fwd(&a, nullptr) != DN_OK) fail(dn_last_error());
    if (teams != c.teams || lone != c.lone || carries != c.carries)
      fail("segment kernels of S " + std::to_string(c.S) + " H " + std::to_string(c.H) + " V " +
           std::to_string(c.V) + ": teams " + std::to_string(teams) + " lone " +
           std::to_string(lone) + " carries " + std::to_string(carries));
  }
  std::printf("ok segment_kernels\n");
}

// The workgroups a whole scan is given, by how many of them the device holds:
// threads of teams (4 waves a team and 4 that stage) or of lone waves.
void scan_shapes() {
  static int team_threads, lone_threads;
  on_launch = [](const Launch& l) {
    if (l.kernel.find("team_scan_kernel") != std::string::npos) team_threads = l.threads;
    if (l.kernel.find("mfma_scan_kernel") != std::string::npos) lone_threads = l.threads;
  };
  const struct {
    int H, K, V, teams, waves;
  } cases[] = {{16, 128, 256, 1, 0}, {17, 128, 256, 2, 0}, {32, 128, 256, 2, 0}, {48, 128, 256, 0, 4},
               {65, 128, 256, 0, 8}, {96, 128, 256, 0, 8}, {64, 64, 64, 1, 0},   {65, 64, 64, 2, 0},
               {129, 64, 64, 0, 4},  {300, 64, 64, 2, 0},  {350, 64, 64, 0, 4},  {129, 64, 128, 0, 8}, {96, 64, 192, 2, 0},
               {128, 64, 192, 0, 4},
               {4, 256, 128, 0, 8}};
  for (const auto& c : cases) {
    dn_chunk_fwd_args a = forward(1, 100, c.H, c.K, c.V, false);
    a.workspace_bytes = dn_chunk_fwd_workspace_bytes(&a);
    team_threads = lone_threads = 0;
    if (dn_chunk_fwd(&a, nullptr) != DN_OK) fail(dn_last_error());
    if (team_threads != (c.teams ? 256 * c.teams + 256 : 0) || lone_threads != 64 * c.waves)
      fail("scan shape of H " + std::to_string(c.H) + " K " + std::to_string(c.K) + " V " +
           std::to_string(c.V) + ": team threads " + std::to_string(team_threads) +
           ", lone threads " + std::to_string(lone_threads));
  }
  std::printf("ok scan_shapes\n");
}

// dn_chunk_bwd where its launches fail one by one: what it left on the second
// stream is joined whenever it returns.
void backward_joins() {
  on_launch = nullptr;
  const struct {
    int dtype, S, H, K, V;
    bool channel;
  } cases[] = {{DN_F32, 130, 2, 64, 64, false},     {DN_BF16, 130, 2, 128, 128, false},
               {DN_BF16, 130, 2, 128, 128, true},   {DN_BF16, 130, 2, 256, 128, false},
               {DN_BF16, 130, 96, 128, 256, false}, {DN_BF16, 130, 2, 64, 64, false}};
  for (const auto& c : cases) {
    dn_chunk_bwd_args a{};
    a.batch = 1, a.sequence = c.S, a.nheads = c.H, a.head_k_dim = c.K, a.head_v_dim = c.V;
    a.erase_width = a.decay_width = c.channel ? c.K : 1;
    a.write_width = c.channel ? c.V : 1;
    a.has_gate = 1, a.chunk_len = 64, a.scale = std::nan("");
    a.qkv_dtype = a.grad_dtype = c.dtype;
    void* const t = const_cast<void*>(kTensor);
    float* const f = static_cast<float*>(t);
    a.d_y = a.q = a.k = a.v = t;
    a.erase = a.write = a.g = a.state_in = f;
    a.d_q = a.d_k = a.d_v = t;
    a.d_erase = a.d_write = a.d_g = a.d_state = f;
    a.workspace = kWorkspace;
    a.workspace_bytes = dn_chunk_bwd_workspace_bytes(&a);
    launches = failing = forks = joins = 0;
    if (dn_chunk_bwd(&a, nullptr) != DN_OK) fail(dn_last_error());
    const int all = launches;
    if (all < 4 || forks != 1 || joins != 1) fail("backward: one fork and one join");
    for (int n = 1; n <= all; ++n) {
      launches = forks = joins = 0;
      failing = n;
      if (dn_chunk_bwd(&a, nullptr) != DN_ERR_HIP) fail("backward: a failed launch is reported");
      if (launches != n) fail("backward: nothing is launched after a failure");
      if (forks != joins)
        fail("backward of K " + std::to_string(c.K) + " dtype " + std::to_string(c.dtype) +
             ": launch " + std::to_string(n) + " of " + std::to_string(all) +
             " failed, and the second stream was not joined");
    }
    failing = 0;
  }
  std::printf("ok backward_joins\n");
}

}  // namespace

int main() {
  out_norm_fallback();
  smaller_workspaces();
  segment_kernels();
  scan_shapes();
  backward_joins();
  std::printf("all passed\n");
  return 0;
}
