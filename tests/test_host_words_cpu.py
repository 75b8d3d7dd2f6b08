"""Error words and counts that calls bring back, on a stand-in for the HIP runtime that runs on the CPU:
host memory for device memory, every launch skipped except the kernel that hands words to the host. With
its pinned memory and, where that can't be had, by plain copies; and for a plan on another device than
the current one, whose memory a kernel of the current device must not read.
"""

import os
import subprocess
import sys

import pytest

RUNTIME = r"""
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

int standin_device = 0, standin_pinned = 1, standin_foreign_reads = 0, standin_copies = 0, standin_published = 0;
static const void *publish;
typedef struct { uint32_t x, y, z; } dim3_;
static struct { dim3_ g, b; size_t sh; void *st; } cfg;

void **__hipRegisterFatBinary(const void *p) { static void *h; (void)p; return &h; }
void __hipUnregisterFatBinary(void **h) { (void)h; }
void __hipRegisterVar(void **h, void *v, char *a, char *b, int c, size_t d, int e, int f) { (void)h; (void)v; (void)a; (void)b; (void)c; (void)d; (void)e; (void)f; }
void __hipRegisterFunction(void **h, const void *f, char *df, const char *name, unsigned n, void *a, void *b, void *c, void *d, int *e)
{
    (void)h; (void)df; (void)n; (void)a; (void)b; (void)c; (void)d; (void)e;
    if (strstr(name, "publish_words_kernel"))
        publish = f;
}
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t sh, void *st) { cfg.g = g; cfg.b = b; cfg.sh = sh; cfg.st = st; return 0; }
int __hipPopCallConfiguration(dim3_ *g, dim3_ *b, size_t *sh, void **st) { *g = cfg.g; *b = cfg.b; *sh = cfg.sh; *st = cfg.st; return 0; }

/* publish_words_kernel(src, n, any, slot, ticket) */
int hipLaunchKernel(const void *f, dim3_ g, dim3_ b, void **args, size_t sh, void *st)
{
    (void)g; (void)b; (void)sh; (void)st;
    if (f != publish)
        return 0;
    if (standin_device != 0) {             /* all memory here is device 0's */
        standin_foreign_reads++;
        return 0;
    }
    const uint32_t *src = *(const uint32_t **)args[0];
    int64_t n = *(int64_t *)args[1], i;
    uint32_t *slot = *(uint32_t **)args[3];
    if (*(unsigned char *)args[2]) {
        slot[0] = 0;
        for (i = 0; i < n; i++)
            slot[0] |= src[i];
    }
    else
        memcpy(slot, src, 4 * n);
    slot[15] = *(uint32_t *)args[4];
    standin_published++;
    return 0;
}
int hipHostMalloc(void **p, size_t n, unsigned fl) { (void)fl; *p = standin_pinned ? calloc(1, n) : 0; return *p ? 0 : 2; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st) { (void)kind; (void)st; memcpy(d, s, n); standin_copies++; return 0; }
int hipStreamSynchronize(void *st) { (void)st; return 0; }
int hipStreamIsCapturing(void *st, int *status) { (void)st; *status = 0; return 0; }
int hipThreadExchangeStreamCaptureMode(int *m) { (void)m; return 0; }
int hipGetLastError(void) { return 0; }
const char *hipGetErrorString(int e) { (void)e; return "error"; }
int hipGetDevice(int *d) { *d = standin_device; return 0; }
int hipPointerGetAttributes(int *a, const void *p) { (void)p; a[0] = 2; a[1] = 0; return 0; }
"""

PROGRAM = r"""
import ctypes, sys
lib_path, runtime, pinned, n = sys.argv[1], sys.argv[2], int(sys.argv[3]), int(sys.argv[4])
rt = ctypes.CDLL(runtime)
word = lambda name: ctypes.c_int.in_dll(rt, "standin_" + name)
word("pinned").value = pinned
lib = ctypes.CDLL(lib_path)
lib.gmm_last_error.restype = ctypes.c_char_p
p, i64, i32 = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int32

class Info(ctypes.Structure):
    _fields_ = [("nsamp", i64), ("ny", i64), ("nx", i64), ("periodic", i32), ("plan_nbytes", i64), ("tmp_nbytes", i64),
                ("overhead", ctypes.c_double), ("ncl", i64), ("nblocks", i64), ("nmt_tb", i64), ("pblocks", i64),
                ("nmt", i64), ("cub", i64), ("max_nchunks", i64)]

def aligned(nbytes):
    b = (ctypes.c_uint8 * (nbytes + 128))()
    a = (ctypes.addressof(b) + 127) & ~127
    keep.append(b)
    return a

keep = []
words = lambda addr, k: (ctypes.c_uint32 * k).from_address(addr)
null = p(None)
xp, err, nmt = aligned(12 * n), aligned(4096), aligned(4096)

# A preplan's three words: error bits and the 64-bit number of entries (here 1).
pre = p()
words(err, 3)[:] = [1, 1, 0]
create = lambda: lib.gmm_preplan_create(ctypes.byref(pre), p(xp), i64(n), i64(64), i64(64), p(nmt), p(err), 0, 0, null)
assert create() != 0 and b"y-value" in lib.gmm_last_error()
words(err, 3)[:] = [0, 1, 0]
assert create() == 0, lib.gmm_last_error()
info = Info()
assert lib.gmm_preplan_get_info(pre, ctypes.byref(info)) == 0
assert info.nmt == 1, info.nmt

plan = p()
buf, tmp = aligned(info.plan_nbytes), aligned(info.tmp_nbytes)
assert lib.gmm_plan_create(ctypes.byref(plan), pre, p(xp), i64(n), p(buf), i64(info.plan_nbytes), p(tmp),
                           i64(info.tmp_nbytes), 0, null) == 0, lib.gmm_last_error()

# The plan's error word follows the planner's (at 128, after one 8-byte entry), on device 0, which is
# current or not.
flag = words(buf + 128 + 4 * info.nblocks, 1)
for device in (0, 1):
    word("device").value = device
    assert lib.gmm_plan_check_errflags(plan, b"check") == 0, lib.gmm_last_error()
    flag[0] = 2
    assert lib.gmm_plan_check_errflags(plan, b"check") != 0, f"error word not seen, device {device} current"
    assert b"check: xpointing x-value" in lib.gmm_last_error()
    assert flag[0] == 0 and lib.gmm_plan_check_errflags(plan, b"check") == 0
word("device").value = 0

# A plan-free call's words, one per block.
off = (i64 * 1)(0)
lp = p()
assert lib.gmm_lpix_create(ctypes.byref(lp), i64(64), i64(64), off, off, i64(1), i64(1), i64(64), i64(4096), 0) == 0
m, tod, nerr = aligned(3 * 4096 * 4), aligned(4 * n), 2048
flags = aligned(4 * nerr)
free = lambda: lib.gmm_unplanned_map2tod(p(tod), i64(n), p(m), i64(3 * 4096), p(xp), i64(n), lp, p(flags), i64(nerr), 0, 0, 1, null)
assert free() == 0, lib.gmm_last_error()
nblocks = (n + 255) // 256
for k in (0, nblocks // 2, nblocks - 1):
    words(flags, nerr)[k] = 1
    assert free() != 0 and b"y-value" in lib.gmm_last_error(), k
    words(flags, nerr)[k] = 0

assert word("foreign_reads").value == 0
assert (word("published").value > 0) == bool(pinned) and word("copies").value > 0
print("ok")
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    d = tmp_path_factory.mktemp("standin")
    (d / "runtime.c").write_text(RUNTIME)
    so = str(d / "libstandin.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", so, str(d / "runtime.c")], check=True)
    return so


@pytest.mark.parametrize("n", [1, 300000])
@pytest.mark.parametrize("pinned", [1, 0])
def test_words(runtime, pinned, n):
    from gpu_mm_amd import _native
    env = dict(os.environ, LD_PRELOAD=":".join([runtime] + os.environ.get("LD_PRELOAD", "").split()))
    r = subprocess.run([sys.executable, "-c", PROGRAM, _native.lib_path(), runtime, str(pinned), str(n)], env=env,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout
