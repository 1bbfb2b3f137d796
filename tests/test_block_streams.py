"""Order and events of the MoE block's two streams (csrc/block.hip), compiled with the host compiler over recorded stand-ins of
the HIP calls and the launches: what the fork waits for is everything that the caller's stream holds by then, host and peer
copies of weights among it, so its event makes the system-wide fence of a plain one; the join orders kernels of one device."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "llmxabe_amd", "csrc")

PROGRAM = r"""
#include <stdio.h>
#include <stdlib.h>
#include "block.hip"

static int streams, events, failing;
static unsigned flags_of[8];
static const char* stream_name(void* s) { return s == (void*)0x100 ? "caller" : s == (void*)0x201 ? "side" : "?"; }
static int step(const char* what, void* s) { printf("%s %s\n", what, stream_name(s)); return XABE_OK; }

extern "C" {
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)(size_t)(0x201 + streams++); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned flags) {
  flags_of[events] = flags;
  *e = (hipEvent_t)(size_t)(0x300 + events++);
  return hipSuccess;
}
static void event(const char* what, hipEvent_t e, hipStream_t s) {
  const int i = (int)((size_t)e - 0x300);
  printf("%s event%d %s%s\n", what, i, stream_name(s), flags_of[i] & hipEventDisableSystemFence ? " device" : " system");
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { event("record", e, s); return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) { event("wait", e, s); return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { *p = malloc(n); return hipSuccess; }
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
int xabe_moe_kernels_new(const xabe_moe_geometry*, xabe_moe_kernels** k) { *k = new xabe_moe_kernels(); return XABE_OK; }
int xabe_moe_buffers_new(const xabe_moe_kernels*, void*, xabe_moe_buffers** b) {
  *b = new xabe_moe_buffers();
  (*b)->x_h = (uint16_t*)0x1000;
  return XABE_OK;
}
int xabe_moe_set_valid_tokens(const xabe_moe_kernels*, void*, xabe_moe_buffers*, size_t) { return XABE_OK; }
int xabe_moe_kernels_tensor_cores_enabled(const xabe_moe_kernels*) { return 1; }
size_t xabe_expert_quant_block_elements(int) { return 32; }
size_t xabe_expert_quant_block_bytes(int) { return 34; }
int xabe_moe_route_and_dispatch(const xabe_moe_kernels*, void* s, xabe_moe_buffers*, const float*, size_t) { return step("route", s); }
int xabe_moe_grouped_forward_partial(const xabe_moe_kernels*, void* s, xabe_moe_buffers*, xabe_quant_tensor, xabe_quant_tensor,
                                     xabe_quant_tensor, const float*, size_t) { return step("routed", s); }
int xabe_moe_shared_expert_mma(const xabe_moe_kernels*, void* s, xabe_moe_buffers*, xabe_quant_tensor, xabe_quant_tensor, xabe_quant_tensor,
                               const float*, size_t, float*, size_t) {
  if (failing) return XABE_ERR_MMA;
  return step("shared", s);
}
int xabe_moe_gate_and_combine(const xabe_moe_kernels*, void* s, const xabe_moe_buffers*, const float*, const float*, const float*, const float*,
                              float*, float*, float*, float*) { return step("combine", s); }
}
namespace xabe {
int set_error(int status, const char*, ...) { return status; }
int hip_error(hipError_t, const char*) { return XABE_ERR_DRIVER; }
bool decode_block_supported(const xabe_moe_kernels*, const xabe_moe_buffers*, const xabe_moe_layer_weights*) { return false; }
bool mfma_supported(const xabe_moe_kernels*, const xabe_moe_buffers*, int, int, int, bool) { return true; }
bool grouped_forward_takes_shared(const xabe_moe_kernels*, const xabe_moe_buffers*, const xabe_moe_layer_weights*) { return false; }
int rms_norm_rows_with_f16(void* s, const float*, const float*, float*, void*, size_t, size_t, float, bool* done) {
  *done = true;
  return step("norm", s);
}
int router_logits_biased(const xabe_moe_kernels*, void* s, const xabe_moe_buffers*, const void*, size_t, int, const float*, size_t,
                         float*, size_t, const float*, bool*, bool*) { return step("router", s); }
}

extern "C" int passes(int refuse) {
  failing = refuse;
  const xabe_moe_geometry g = {8, 2, 512, 256, 32, 64};
  xabe_moe_block* blk = nullptr;
  void* caller = (void*)0x100;
  if (xabe_moe_block_new(&g, 1e-6f, caller, &blk) != XABE_OK) return 1;
  xabe_moe_layer_weights w = {};
  w.router_quant = -1;
  float x = 0.0f;
  const size_t n = 64 * 512;
  const int st = xabe_moe_block_forward(blk, caller, &w, &x, n, 64, nullptr, &x, n, &x, n);
  printf("status %s\n", st == XABE_OK ? "ok" : "error");
  return 0;
}
"""

# (bound as they are called: what the forward of this program does not reach stays undefined)
RUNNER = r"""
#include <dlfcn.h>
int main(int argc, char** argv) {
  void* lib = dlopen(argv[1], RTLD_LAZY);
  return lib ? reinterpret_cast<int (*)(int)>(dlsym(lib, "passes"))(argc > 2) : 1;
}
"""


@pytest.fixture(scope="module")
def steps(tmp_path_factory):
    d = tmp_path_factory.mktemp("streams")
    (d / "streams.cpp").write_text(PROGRAM)
    (d / "runner.cpp").write_text(RUNNER)
    subprocess.check_call(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-w", "-I/opt/rocm/include", "-I", CSRC, "-shared", "-fPIC", "-Wl,-z,lazy",
                           str(d / "streams.cpp"), "-o", str(d / "streams.so")])
    subprocess.check_call(["g++", str(d / "runner.cpp"), "-o", str(d / "runner"), "-ldl"])

    def run(*args):
        r = subprocess.run([str(d / "runner"), str(d / "streams.so"), *args], capture_output=True, text=True)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout.splitlines()

    return run


def test_fork_and_join_enclose_the_side_streams_work(steps):
    assert steps() == ["norm caller", "record event0 caller system", "wait event0 side system", "shared side", "record event1 side device",
                       "router caller", "route caller", "routed caller", "wait event1 caller device", "combine caller", "status ok"]


def test_a_refused_shared_expert_is_joined_all_the_same(steps):
    assert steps("refuse") == ["norm caller", "record event0 caller system", "wait event0 side system", "record event1 side device",
                               "wait event1 caller device", "status error"]
