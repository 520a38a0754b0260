"""Where a product's workspace comes from: abi.cpp against a stand-in HIP runtime
in which allocations fail and another handle's scratch work stays pending on
demand. CPU only."""
from __future__ import annotations

import subprocess

import pytest

from conftest import PACKAGE_DIR, ROOT

# The stand-in keeps the last error as HIP does until it is asked for; a launch
# reports it as its own.
SOURCE = r"""
#include "abi.cpp"
#include <cstdio>

static hipError_t last = hipSuccess;
static bool fail_malloc = false, pending = false;
static ackvq::MatmulPath path = ackvq::MatmulPath::General;
static size_t need = 0;
static int launches = 0;
static void* launch_work = nullptr;
static size_t launch_bytes = 0;

extern "C" {
hipError_t hipGetLastError() { hipError_t e = last; last = hipSuccess; return e; }
hipError_t hipMalloc(void** p, size_t n) {
  if (fail_malloc) return last = hipErrorOutOfMemory;
  *p = std::malloc(n < 64 ? n : 64);
  return hipSuccess;
}
hipError_t hipFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipMemset(void*, int, size_t) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600*, int) { return hipErrorInvalidValue; }
hipError_t hipDeviceGetName(char* s, int, int) { s[0] = 'x'; s[1] = 0; return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)1; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)1; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return pending ? (last = hipErrorNotReady) : hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void* s) { *p = const_cast<void*>(s); return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
}
namespace ackvq {
MatmulPath choose_matmul_path(uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t) { return path; }
MatmulPath choose_dense_path(uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t) { return path; }
size_t matmul_workspace_bytes(MatmulPath, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t) { return need; }
size_t dense_workspace_bytes(MatmulPath, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t) { return need; }
static hipError_t launched(MatmulPath p, void* work, size_t bytes) {
  ++launches;
  path = p;
  launch_work = work;
  launch_bytes = bytes;
  return hipGetLastError();
}
hipError_t launch_matmul(hipStream_t, const Operands&, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t,
                         MatmulPath p, void* work, size_t bytes) { return launched(p, work, bytes); }
hipError_t launch_matmul_dense(hipStream_t, const Operands&, uint32_t, uint32_t, uint32_t, uint32_t,
                               uint32_t, MatmulPath p, void* work, size_t bytes) { return launched(p, work, bytes); }
}

static int failures = 0;
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s (%s)\n", __LINE__, #x, text()); ++failures; } } while (0)
static const char* text() {
  static char s[256];
  s[0] = 0;
  ack_last_error(s, sizeof s);
  return s;
}

struct Handle {
  AckDevice* dev = ack_open();
  AckBuffer* b[6];
  Handle() { for (auto& x : b) x = ack_buffer_alloc(dev, 1 << 20); }
  int run(const char* entry) {
    const uint32_t words[8] = {2, 64, 64, 64, 16, 16, 0, 0};
    const uint8_t* plan = reinterpret_cast<const uint8_t*>(words);
    if (entry[0] == 'n') return ack_vq_noalloc(dev, b[0], b[1], b[2], b[3], b[4], b[5], plan, 32);
    if (entry[0] == 'd') return ack_vq_matmul_dense(dev, b[0], b[2], b[3], b[4], b[5], plan, 32);
    return ack_vq(dev, b[0], b[1], b[2], b[3], b[4], b[5], plan, 32);
  }
};

int main(int argc, char** argv) {
  using P = ackvq::MatmulPath;
  const P optional[] = {P::GeneralMfma, P::GramMfma, P::JointMfma};
  const std::string which = argv[1];
  Handle one, two;
  if (which == "memory") {
    // a full GPU: optional workspaces are done without, and nothing reports an error
    for (P p : optional)
      for (const char* entry : {"vq", "dense"}) {
        path = p, need = size_t(4) << 20, fail_malloc = true;
        const int before = launches;
        CHECK(one.run(entry) == ACK_OK);
        CHECK(launches == before + 1 && path == p && launch_work == nullptr);
        CHECK(last == hipSuccess && text()[0] == 0);
        fail_malloc = false;
      }
    // a path that needs its workspace reports the failure, and only that call does
    path = P::OneHotMfma, fail_malloc = true;
    const int before = launches;
    CHECK(one.run("vq") == ACK_ERR_DEVICE && launches == before);
    fail_malloc = false;
    CHECK(one.run("vq") == ACK_OK && launch_work != nullptr && last == hipSuccess);
  } else {
    // noalloc: one handle's pending scratch work refuses the other's, and neither
    // is in the way of the optional paths, nor they of it
    path = P::OneHotMfma, need = 4096, pending = true;
    CHECK(one.run("noalloc") == ACK_OK);
    for (P p : optional)
      for (size_t bytes : {size_t(0), size_t(4) << 20, size_t(12) << 20, size_t(100) << 20}) {
        path = p, need = bytes;
        // joint-mfma's codes past the scratch's size: the general kernel, by size alone
        const bool general = p == P::JointMfma && bytes > size_t(16) << 20;
        CHECK(two.run("noalloc") == ACK_OK && path == (general ? P::General : p));
        CHECK(bytes <= size_t(8) << 20 ? launch_work != nullptr && launch_bytes == bytes
                                       : general || launch_work == nullptr);
        path = p;
        CHECK(one.run("noalloc") == ACK_OK);
      }
    path = P::OneHotMfma, need = 4096;
    CHECK(two.run("noalloc") == ACK_ERR_DEVICE && path == P::OneHotMfma);
    CHECK(one.run("noalloc") == ACK_OK);
    need = size_t(17) << 20;
    CHECK(one.run("noalloc") == ACK_ERR_SIZE);
    need = 4096, pending = false;
    CHECK(two.run("noalloc") == ACK_OK);
  }
  return failures != 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    folder = tmp_path_factory.mktemp("abi")
    source, out = folder / "workspace.cpp", folder / "workspace"
    source.write_text(SOURCE)
    subprocess.run(
        ["g++", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-DACK_SHADERS_ID=1ull",
         "-D__align__(x)=__attribute__((aligned(x)))", "-DHIP_SYMBOL(x)=(&x)",
         "-I/opt/rocm/include", f"-I{ROOT / 'include'}", f"-I{PACKAGE_DIR / 'csrc'}", str(source),
         "-o", str(out), "-Wl,--unresolved-symbols=ignore-all"], check=True)
    return out


@pytest.mark.parametrize("which", ["memory", "scratch"])
def test_workspace(program, which):
    done = subprocess.run([str(program), which], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stdout + done.stderr
