"""What the host does in a call of the fused MLP, on the CPU: the library is loaded in a process of its own beside a stand-in for the few functions of the HIP
runtime that it calls, which counts device look-ups and records the launches and carries out nothing."""
import ctypes
import json
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

RUNTIME = r"""
#include <stddef.h>
typedef struct { unsigned x, y, z; } dim3_;
static dim3_ g, b; static size_t lds; static void* st;
int lookups, launches, threads[256], blocks[256], bytes[256];
int hipGetDevice(int* d) { *d = 0; ++lookups; return 0; }
int hipDeviceGetAttribute(int* v, int attr, int dev) { (void)attr; (void)dev; *v = 256; return 0; }
int hipFuncSetAttribute(const void* f, int a, int v) { (void)f; (void)a; (void)v; return 0; }
int hipGetLastError(void) { return 0; }
int __hipPushCallConfiguration(dim3_ grid, dim3_ block, size_t shmem, void* stream) { g = grid; b = block; lds = shmem; st = stream; return 0; }
int __hipPopCallConfiguration(dim3_* grid, dim3_* block, size_t* shmem, void** stream) { *grid = g; *block = b; *shmem = lds; *stream = st; return 0; }
int hipLaunchKernel(const void* f, dim3_ grid, dim3_ block, void** args, size_t shmem, void* stream)
{
    (void)f; (void)args; (void)stream;
    if (launches < 256) { blocks[launches] = grid.x; threads[launches] = block.x; bytes[launches] = (int)shmem; }
    ++launches;
    return 0;
}
"""

# arguments: stand-in, library, sizes as JSON; prints look-ups of the workspace query and, per pass, look-ups and the launches' {workgroups, threads, LDS}
CHILD = r"""
import ctypes, json, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
P, L, I, F, Z = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int, ctypes.c_float, ctypes.c_size_t
lib.moe_mlp_workspace_bytes.restype = Z
lib.moe_mlp_workspace_bytes.argtypes = [L, I, L, L, I]
lib.moe_mlp_fwd.argtypes = [P, L, P, P, P, P, P, I, F, P, P, P, P, L, P, I, P, I, I, L, L, L, I, I, I, P, P, Z, P]
lib.moe_mlp_bwd.argtypes = [P, L, I, I, P, P, L, P, P, P, P, P, P, P, I, F, P, P, P, P, P, P, L, I, P, I, P, I, I, L, L, L, I, I, P, P, Z, P]
def val(n): return ctypes.c_int.in_dll(fake, n)
def arr(n): return (ctypes.c_int * 256).in_dll(fake, n)
out = []
for R, E, d, f, r in json.loads(sys.argv[3]):
    val("lookups").value = 0
    n = lib.moe_mlp_workspace_bytes(R, E, d, f, r)
    res = {"query": val("lookups").value, "bytes": n}
    one = 256   # a stand-in for every pointer: nothing here dereferences one
    lora = (P * 6)(*[one] * 6) if r else None
    st = (L * 18)(*[1] * 18) if r else None
    def fwd(): return lib.moe_mlp_fwd(one, d, one, one, one, lora, st, r, 1.0, one, one, one, one, d, one, 0, one, 0, E, R, d, f, 2, 0, 0, one, one, n, None)
    def bwd(): return lib.moe_mlp_bwd(one, d, 0, 1, one, one, d, one, one, one, lora, st, lora, st, r, 1.0, one, one, one, one, one, one, d, 0, one, 0, one, 0, E, R, d, f, 2, 0, one, one, n, None)
    for name, call in (("fwd", fwd), ("bwd", bwd)):
        val("lookups").value = val("launches").value = 0
        rc = call()
        k = val("launches").value
        res[name] = {"rc": rc, "lookups": val("lookups").value, "launches": [[arr(a)[i] for a in ("blocks", "threads", "bytes")] for i in range(k)]}
    out.append(res)
print(json.dumps(out))
"""


@pytest.fixture(scope="module")
def calls(tmp_path_factory):
    from moe_distributed_training_amd._lib import LIB_PATH
    cc = shutil.which("cc") or shutil.which("gcc")
    if cc is None:
        pytest.skip("no C compiler")
    tmp = tmp_path_factory.mktemp("runtime")
    (tmp / "runtime.c").write_text(RUNTIME)
    so = str(tmp / "runtime.so")
    subprocess.run([cc, "-shared", "-fPIC", "-O1", "-o", so, str(tmp / "runtime.c")], check=True)

    def run(*sizes):
        p = subprocess.run([sys.executable, "-c", CHILD, so, LIB_PATH, json.dumps(sizes)], capture_output=True, text=True, timeout=120)
        assert p.returncode == 0, p.stderr[-2000:]
        return json.loads(p.stdout)
    return run


@pytest.mark.parametrize("R,E,d,f,r", [(1024, 8, 256, 512, 16), (1024, 8, 256, 512, 0), (100, 2, 1024, 512, 16), (8192, 8, 4096, 14336, 16), (2, 8, 4096, 14336, 0), (1024, 8, 256, 512, 64)])
def test_a_pass_looks_the_device_up_once_and_per_launch(calls, R, E, d, f, r):
    """The tile choice and the areas that depend on it come from one plan: the workspace query looks the device up once, a pass once and at most twice for each launch
    (its dynamic LDS is allowed per device; some count compute units for their grid)."""
    res, = calls((R, E, d, f, r))
    assert res["query"] == 1
    for name in ("fwd", "bwd"):
        assert res[name]["rc"] == 0 and res[name]["launches"]
        assert res[name]["lookups"] <= 1 + 2 * len(res[name]["launches"]), (name, res[name]["lookups"], len(res[name]["launches"]))


# rows, groups, d, f: what the host sees of launches whose small tiles came to more than the compute units where rows are not dealt evenly
UNEVEN = [(253, 2, 4096, 14336), (1988, 16, 896, 1856), (3934, 32, 512, 896), (7768, 64, 192, 1408), (2248, 16, 768, 1216), (975, 8, 1728, 1856), (1992, 16, 2816, 960), (3617, 1, 704, 1472)]
EVEN = [(1024, 8, 256, 512), (2, 8, 4096, 14336), (64, 1, 4096, 14336), (200, 4, 512, 2048), (17, 16, 1024, 512)]


@pytest.mark.parametrize("r", [0, 16])
def test_small_tiles_however_the_rows_fall(calls, r):
    """A launch that may split K takes tiles of 128 x 128 (4 waves, 80 KiB of LDS) only where these come to at most one per compute unit for any group sizes, one that never splits up to one and
    a half; groups of a row more than 128 are two small tiles and one large one, and from there on the small ones were slower, by up to a quarter."""
    sizes = UNEVEN + EVEN
    small_seen = 0
    for (R, E, d, f), res in zip(sizes, calls(*[(*s, r) for s in sizes])):
        gemms = {n: [l for l in res[n]["launches"] if l[2] >= 80 * 1024] for n in ("fwd", "bwd")}
        assert [len(gemms["fwd"]), len(gemms["bwd"])] == [2, 2]
        groups = min(R, E)
        rows = groups + (R - groups) // 128   # tiles of 128 rows, at most
        for (_, threads, lds), K, N, pair in zip(gemms["fwd"] + gemms["bwd"], (d, f, d, 2 * f), (f, d, f, d), (True, False, False, False)):
            assert (threads, lds) in ((256, 80 * 1024), (512, 160 * 1024))
            parts = 1 if pair else next(p for p in (4, 2, 1) if p == 1 or K // 64 // p >= 8)
            tiles = rows * -(-N // (64 if pair else 128)) * parts
            if threads == 256:
                assert 2 * tiles <= (2 if parts > 1 else 3) * 256, (R, E, d, f, K, N, pair, tiles)
                small_seen += 1
        if (R, E, d, f) in EVEN[:2]:   # (what small tiles are for: a narrow layer, one token of the wide one)
            assert gemms["fwd"][1][1] == 256 and gemms["bwd"][1][1] == 256
    assert small_seen >= 12
