"""A child process in which the library's calls of the HIP runtime pass through a few hooks, so that a
test can refuse one from the host (no pinned memory, a launch that fails) or count them.  A refused
call never reaches the runtime."""
import os
import subprocess
import sys
import textwrap

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HOOKS = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
#include <unistd.h>
typedef struct { unsigned x, y, z; } Dim;
enum { OUT_OF_MEMORY = 2, LAUNCH_FAILURE = 719 };
int hook_pinned_left = 1 << 30; /* hipHostMalloc calls that still succeed */
int hook_fail_launches = 0;     /* launches refused from now on */
int hook_copies = 0;            /* hipMemcpyAsync calls */
static __thread int pending, slow;
static void* real(const char* name)
{
    static void* lib;
    if (!lib) lib = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
    return dlsym(lib, name);
}
int hipHostMalloc(void** p, size_t n, unsigned flags)
{
    if (__sync_fetch_and_sub(&hook_pinned_left, 1) <= 0) {
        pending = OUT_OF_MEMORY;
        return OUT_OF_MEMORY;
    }
    return ((int (*)(void**, size_t, unsigned))real("hipHostMalloc"))(p, n, flags);
}
int hipLaunchKernel(const void* f, Dim grid, Dim block, void** args, size_t lds, void* stream)
{
    if (hook_fail_launches > 0) {
        hook_fail_launches--;
        pending = LAUNCH_FAILURE;
        slow = 1;
        return LAUNCH_FAILURE;
    }
    return ((int (*)(const void*, Dim, Dim, void**, size_t, void*))real("hipLaunchKernel"))(f, grid, block, args, lds, stream);
}
int hipGetLastError(void)
{
    const int e = pending;
    pending = 0;
    return e ? e : ((int (*)(void))real("hipGetLastError"))();
}
int hipSetDevice(int d) /* held up after a refused launch, so that other threads come first */
{
    if (slow) usleep(500000);
    slow = 0;
    return ((int (*)(int))real("hipSetDevice"))(d);
}
int hipMemcpyAsync(void* to, const void* from, size_t n, int kind, void* stream)
{
    __sync_fetch_and_add(&hook_copies, 1);
    return ((int (*)(void*, const void*, size_t, int, void*))real("hipMemcpyAsync"))(to, from, n, kind, stream);
}
"""

PRELUDE = """
import ctypes, sys
hooks = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path[:0] = [sys.argv[2], sys.argv[2] + "/tests"]
import numpy as np
import ziran2020_amd
from ziran2020_amd import _abi as A, scenes
gpu = ziran2020_amd.load_library()
def hook(name):
    return ctypes.c_int.in_dll(hooks, "hook_" + name)
"""


def run(tmp_path, body, *args):
    """The statements of `body` in the child (args are its sys.argv[3:]); fails if it does."""
    src, lib = tmp_path / "hooks.c", tmp_path / "hooks.so"
    src.write_text(HOOKS)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", str(src), "-o", str(lib), "-ldl"], check=True)
    out = subprocess.run([sys.executable, "-u", "-c", PRELUDE + textwrap.dedent(body), str(lib), ROOT, *map(str, args)],
                         capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stdout[-2000:] + out.stderr[-4000:]
