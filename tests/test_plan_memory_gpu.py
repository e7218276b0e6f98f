"""Transcode plans when device memory is short: a plan whose four-block tables
do not fit is built with the smaller two-block ones and decodes as ever, and a
call that runs out of memory leaves nothing behind for the next one.

Allocations fail in a child process whose hipMalloc is a wrapper around the
runtime's: above a size it asks the runtime for 2^50 bytes instead, so that the
runtime itself refuses and keeps the error as it does for any other refusal."""
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

WRAPPER = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
size_t fail_above = (size_t)-1;
int failed = 0;
int hipMalloc(void** p, size_t n)
{
    static int (*real)(void**, size_t);
    if (!real) real = (int (*)(void**, size_t))dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD), "hipMalloc");
    if (n > fail_above) {
        failed++;
        n = (size_t)1 << 50;
    }
    return real(p, n);
}
"""

CHILD = r"""
import ctypes as C, sys
wrap = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)   # ahead of every user of the runtime
import numpy as np, torch
import oracle
from crunch2_amd import crnd, texture
from crunch2_amd._lib import FMT_DXT5, lib
above, failed = C.c_size_t.in_dll(wrap, "fail_above"), C.c_int.in_dll(wrap, "failed")
data = texture.synth_crn(512, 5, FMT_DXT5)
bits = 8 * len(data)
ref = oracle.unpack_all(data)
exp = np.concatenate([ref[l][0].reshape(-1) for l in sorted(ref)])
out = torch.zeros(len(exp), dtype=torch.uint8, device="cuda")
levels = len(ref)
stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)


def decode(ctx, first=0, count=levels):
    out.zero_()
    rc = lib().crn2_unpack_levels_device(C.c_void_p(ctx.handle), out.data_ptr(), len(exp), first, count, stream)
    torch.cuda.synchronize()
    return rc


mode = sys.argv[2]
ctx = crnd.unpack_begin(data)
# scratch per stream bit: 20 to 24 bytes with four-block tables, 8 to 10 with two-block
# ones, and under 4 for everything else of this file
above.value = 15 * bits if mode == "tables" else 1 << 16
if mode == "tables":
    assert decode(ctx) == 0 and np.array_equal(out.cpu().numpy(), exp)
    assert failed.value == 1, failed.value
    plan = C.c_void_p()
    handle, dst, size = (C.c_void_p * 1)(ctx.handle), (C.c_void_p * 1)(out.data_ptr()), (C.c_uint64 * 1)(len(exp))
    assert lib().crn2_batch_create(handle, 1, dst, size, C.byref(plan)) == 0 and failed.value == 2
    for run in (lib().crn2_batch_run, lib().crn2_batch_run_graph):
        out.zero_()
        assert run(plan, stream) == 0 and lib().crn2_batch_status(plan, stream) == 0
        assert np.array_equal(out.cpu().numpy(), exp)
    lib().crn2_batch_destroy(plan)
else:
    assert decode(ctx) != 0 and failed.value == 2
    assert crnd.unpack_begin(data) is None
    above.value = (1 << 64) - 1
    assert decode(ctx) == 0 and np.array_equal(out.cpu().numpy(), exp)
assert np.array_equal(crnd.unpack_level(ctx, 1)[0], ref[1][0])
assert crnd.unpack_end(ctx)
print("plan memory ok", failed.value, flush=True)
"""


@pytest.mark.parametrize("mode", ["tables", "all"])
def test_short_of_memory(gpu, tmp_path, mode):
    print("plan memory", mode, flush=True)
    src, so = tmp_path / "wrap.c", tmp_path / "wrap.so"
    src.write_text(WRAPPER)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", str(so), str(src), "-ldl"], check=True)
    r = subprocess.run([sys.executable, "-u", "-c", CHILD, str(so), mode], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "plan memory ok" in r.stdout, r.stdout + r.stderr
