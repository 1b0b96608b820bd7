"""Calls that read back through pinned host memory give the same results where the system has none to give: the read-back
then goes through pageable memory. A shim refuses hipHostMalloc in a child process."""
import subprocess
import sys
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu
SHIM = """
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
static int armed, count;
void arm(int v) { armed = v; }
int refused(void) { return count; }
int hipHostMalloc(void** p, size_t n, unsigned flags) {
  static int (*real)(void**, size_t, unsigned);
  if (armed) { ++count; return 2; }                     /* hipErrorOutOfMemory */
  if (!real) real = (int (*)(void**, size_t, unsigned))dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD), "hipHostMalloc");
  return real(p, n, flags);
}
"""


@pytest.mark.parametrize("call", ["prefill", "bank"])
def test_no_pinned_memory(gpu, tmp_path, call):
    (tmp_path / "shim.c").write_text(SHIM)
    so = tmp_path / "shim.so"
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", str(so), str(tmp_path / "shim.c"), "-ldl"], check=True)
    child = Path(__file__).with_name("pinned_refusal_child.py")
    r = subprocess.run([sys.executable, "-u", str(child), str(so), call], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
