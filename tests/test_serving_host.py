"""Admission control of the serving loop, host side (no GPU): the memory
gate admits a batch while the running estimates fit the budget (any batch
on an idle device), and the estimator follows measured bytes per unit."""
import subprocess
import threading
import time
from pathlib import Path

import gpu_graph_mining_amd as gm
from gpu_graph_mining_amd import build as gbuild
from gpu_graph_mining_amd import serving

ROOT = Path(__file__).resolve().parent.parent


def test_gate_admits_within_budget_and_waits_for_memory():
    gate = serving.MemoryGate(100)
    stop = threading.Event()
    assert gate.admit_first(80, stop)          # idle device: admitted
    assert not gate.admit_more(30)             # 110 > 100
    assert gate.admit_more(20)                 # 100
    admitted = []

    def second():
        admitted.append(gate.admit_first(50, stop))

    t = threading.Thread(target=second)
    t.start()
    time.sleep(0.2)
    assert not admitted                        # waits: 100 + 50 > 100
    gate.release(100)                          # the first batch ends
    t.join(2)
    assert admitted == [True] and gate.used == 50 and gate.running == 1
    gate.release(50)
    assert gate.admit_first(10_000, stop)      # larger than the budget, but alone
    gate.release(10_000)


def test_gate_wait_ends_when_the_server_stops():
    gate = serving.MemoryGate(10)
    stop = threading.Event()
    assert gate.admit_first(10, stop)
    out = []
    t = threading.Thread(target=lambda: out.append(gate.admit_first(5, stop)))
    t.start()
    time.sleep(0.1)
    stop.set()
    t.join(2)
    assert out == [False]


def test_estimator_follows_measurements():
    e = serving.Estimator(16.0)
    r = serving.Request(serving.QUERY, 0, units=1000)
    assert e.estimate(r) == 16001
    e.observe(1000, 64000)                     # 64 bytes per unit measured
    assert e.per_unit >= 32.0                  # never far below the latest
    for _ in range(30):
        e.observe(1000, 64000)
    assert abs(e.per_unit - 64.0) < 1.0
    e.observe(0, 5)                            # nothing measured: unchanged
    assert abs(e.per_unit - 64.0) < 1.0


def test_failed_allocations_free_the_kept_batches_and_try_again(tmp_path):
    """Device and pinned buffers alike: an allocation that fails for want of
    memory frees what is kept for later subset batches and is tried once more;
    any other failure, or nothing kept, is the caller's error.  (No GPU: the
    program's own allocators stand before the runtime's.)"""
    src = tmp_path / "alloc.cpp"
    src.write_text('''#include <cstdio>
#include <cstdlib>
#include "miner.hpp"
static int fails, calls, freed;
static bool kept;
static hipError_t error;
static hipError_t take(void **p, size_t n) {
  ++calls;
  if (fails-- > 0) return error;
  *p = std::malloc(n);
  return hipSuccess;
}
bool gm::release_spares() {
  ++freed;
  return kept;
}
extern "C" {
hipError_t hipMalloc(void **p, size_t n) { return take(p, n); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return take(p, n); }
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void **d, void *p, unsigned) { *d = p; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
}
template <class Buf>
void run(const char *name) {
  for (int f = 0; f < 3; ++f)
    for (int k = 0; k < 2; ++k)
      for (hipError_t e : {hipErrorOutOfMemory, hipErrorInvalidValue}) {
        fails = f;
        kept = k;
        error = e;
        calls = freed = 0;
        int code = 0;
        Buf b;
        try {
          b.ensure(100);
        } catch (const gm::Error &x) {
          code = x.code;
        }
        std::printf("%s %d %d %d : %d %d %d\\n", name, f, k, (int)(e == hipErrorOutOfMemory), calls, freed, code);
      }
}
int main() {
  run<gm::DevBuf>("dev");
  run<gm::HostBuf>("host");
}
''')
    exe = tmp_path / "alloc"
    subprocess.run(["g++", "-std=c++17", "-rdynamic", "-D__HIP_PLATFORM_AMD__", f"-I{ROOT / 'include'}",
                    f"-I{ROOT / 'gpu_graph_mining_amd' / 'csrc'}", "-I/opt/rocm/include", str(src), f"-L{gbuild.LIB_DIR}",
                    "-lgspan_amd", f"-Wl,-rpath,{gbuild.LIB_DIR}", "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout.split("\n")
    want = []
    for name in ("dev", "host"):
        for fails in range(3):
            for kept in range(2):
                for oom in (1, 0):
                    again = fails > 0 and oom and kept
                    calls = 2 if again else 1
                    code = 0 if fails < calls else gm.GM_E_OOM if oom else gm.GM_E_DEVICE
                    want.append(f"{name} {fails} {kept} {oom} : {calls} {int(fails > 0 and oom)} {code}")
    assert out[:-1] == want


def test_kept_batches_take_a_small_share_of_the_budget():
    for budget in (0, 1, 256 << 20, 4 << 30, 8 << 30, 64 << 30, 1 << 40):
        for slots in (1, 2, 4):
            limit, reserve = serving.spare_bytes(budget, slots)
            assert reserve == (slots + 2) * limit <= budget * (slots + 2) // 32
            assert limit == 0 or 128 << 20 <= limit <= 1 << 30
            assert (limit > 0) == (budget >= 4 << 30)
