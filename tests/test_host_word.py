"""The word that a kernel writes and the calling thread waits for (cumm_amd/csrc/host_word.h), with a HIP runtime
of a few lines in its place: the kind of memory, who gets a word again and who does not."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "cumm_amd", "csrc")

# (names and values of the public interface; the rest is what the test looks at)
RUNTIME = r"""
#pragma once
#include <cstdlib>
typedef int hipError_t;
typedef void *hipStream_t;
constexpr int hipSuccess = 0, hipErrorUnknown = 999, hipErrorNotReady = 600;
constexpr unsigned hipHostMallocPortable = 0x1, hipHostMallocCoherent = 0x40000000;
inline int answer = hipErrorNotReady, asked = 0, mallocs = 0;
inline unsigned flags = 0;
inline unsigned *write_when_asked = nullptr;
inline hipError_t hipHostMalloc(void **at, size_t n, unsigned f) { flags = f; ++mallocs; *at = malloc(n); return hipSuccess; }
inline hipError_t hipStreamQuery(hipStream_t) { if (++asked == 2 && write_when_asked) *write_when_asked = 7; return answer; }
inline hipError_t hipGetLastError() { return hipSuccess; }
"""

PROGRAM = r"""
#include "host_word.h"
#include <cstdio>
#define EXPECT(x) do { if (!(x)) { printf("not so: %s (line %d)\n", #x, __LINE__); return 1; } } while (0)
using cummhip::HostWord;
int main() {
  uint32_t v = 0, *first = nullptr, *second = nullptr;
  {
    HostWord w;
    EXPECT(w.take() == hipSuccess && *w.at == cummhip::kNotYet);
    EXPECT((flags & hipHostMallocCoherent) && (flags & hipHostMallocPortable));
    write_when_asked = first = w.at;
    EXPECT(w.wait(nullptr, &v) == hipSuccess && v == 7 && asked == 2);
    HostWord other;                                  // a call in another thread meanwhile
    EXPECT(other.take() == hipSuccess && other.at != first);
    second = other.at;
    answer = hipErrorUnknown;
    EXPECT(other.wait(nullptr, &v) == hipErrorUnknown && !other.settled);
  }
  {
    HostWord w;                                      // the first word again, cleared; not the one whose kernel may still write
    EXPECT(w.take() == hipSuccess && w.at == first && *w.at == cummhip::kNotYet);
    HostWord x;
    EXPECT(x.take() == hipSuccess && x.at != second && mallocs == 3);
    answer = hipSuccess;                             // a launch that ended without writing is no endless wait
    EXPECT(w.wait(nullptr, &v) == hipSuccess && v == cummhip::kNotYet);
  }
  return 0;
}
"""


def test_words_that_a_kernel_writes_and_a_thread_waits_for(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("no host compiler")
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (tmp_path / "main.cpp").write_text(PROGRAM)
    program = str(tmp_path / "main")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", str(tmp_path), "-I", CSRC, str(tmp_path / "main.cpp"), "-o", program], check=True)
    run = subprocess.run([program], stdout=subprocess.PIPE, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
