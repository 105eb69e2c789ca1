"""The C-ABI library loads without a GPU, exports every symbol include/moe_hip.h declares with the signature the
Python binding assumes, and rejects bad arguments before touching the device."""
import ctypes
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _header_decls():
    hdr = open(os.path.join(ROOT, "include", "moe_hip.h")).read()
    hdr = re.sub(r"/\*.*?\*/", "", hdr, flags=re.S)
    decls = {}
    for m in re.finditer(r"\b(moe_\w+)\s*\(([^;{]*?)\)\s*;", hdr, flags=re.S):
        args = m.group(2).strip()
        codes = ""
        for a in ([] if args == "void" else [a.strip() for a in args.split(",")]):
            codes += "p" if "*" in a else "l" if a.startswith("int64_t") else "z" if a.startswith("size_t") else \
                "f" if a.startswith("float") else "i"
        decls[m.group(1)] = codes
    return decls


def test_library_exports_every_declared_symbol():
    from moe_distributed_training_amd import _lib
    decls = _header_decls()
    assert len(decls) >= 25
    raw = ctypes.CDLL(_lib.LIB_PATH)
    for name in decls:
        assert hasattr(raw, name), f"libmoe_hip.so does not export {name}"
    assert set(decls) == set(_lib._SIGNATURES), set(decls) ^ set(_lib._SIGNATURES)
    for name, codes in decls.items():
        assert _lib._SIGNATURES[name][1] == codes, f"binding of {name} disagrees with the header"
    assert _lib.lib.moe_hip_abi_version() == _lib.ABI_VERSION == int(re.search(r"#define\s+MOE_HIP_ABI_VERSION\s+(\d+)", open(os.path.join(ROOT, "include", "moe_hip.h")).read()).group(1))


def test_bad_arguments_are_rejected_on_the_host():
    from moe_distributed_training_amd._lib import lib
    assert lib.moe_hip_strerror(0) == b"ok" and lib.moe_hip_strerror(-3) == b"workspace too small"
    # null pointers / inconsistent sizes: status -1 and nothing is launched
    assert lib.moe_router_topk(None, None, None, None, 4, 8, 2, 1, None) == -1
    assert lib.moe_router_topk(1, 1, 1, 1, 4, 8, 9, 1, None) == -1          # k > E
    assert lib.moe_scatter2scatter(None, 1, 1, None, 1, 1, 1, None, 0, 0, 0, None, 0, 0, 0, 0, 0.0, None, 1, 1, None, 0,
                                   None, 0, 4, 8, 16, 16, 1, 0, 0, 0, None, 0, None) == -1
    assert lib.moe_group_bwd_ab(None, 1, 1, None, 1, 1, None, 1, 1, 1, None, 1, 1, 1, 4, 1.0, None, 1, 1, 1, None, 1, 1, 1,
                                None, 0, 2, 8, 16, 16, 0, None, 0, None) == -1
    assert lib.moe_mlp_fwd(None, 1, None, None, None, None, None, 0, 0.0, None, None, None, None, 1, None, 0, None, 0, 2,
                           8, 64, 64, 1, 0, 0, None, None, 0, None) == -1
    assert lib.moe_sort_workspace_bytes(8192, 8) >= 4 * 8 * 4
    # the sort's status path: more experts than the counting sort takes (4096) is refused before anything is enqueued
    # (16: non-null stand-ins that are never dereferenced); this is what flatten_and_sort's RuntimeError comes from
    assert lib.moe_sort_by_expert(16, 0, 8, 4097, 128, 16, 16, 0, None, None, None, 0, None, None, 16, 1 << 20, None) == -1
    assert lib.moe_sort_by_expert_static(16, 0, 8, 4097, 128, 16, 16, 0, None, None, None, 0, None, None, None) == -1
    assert lib.moe_mlp_workspace_bytes(8192, 8, 4096, 14336, 16) > 0


def test_cpu_tensors_fail_loudly():
    import pytest
    import torch
    import moe_distributed_training_amd as moe
    with pytest.raises(RuntimeError, match="GPU only"):
        moe.flatten_and_sort(torch.tensor([1, 0, 1]))
    with pytest.raises(RuntimeError, match="GPU only"):
        moe.forward_router(torch.randn(4, 8), torch.randn(2, 8), 1)


def test_size_limits_are_checked_before_anything_is_enqueued():
    """The fused entry points address gathered activation rows and one expert's matrix with 32-bit byte offsets; sizes
    beyond that are refused on the host with MOE_ERR_UNSUPPORTED (status codes only: nothing is dereferenced), while the
    number of rows alone never is (grouped tiles are addressed from their own first row)."""
    from moe_distributed_training_amd._lib import lib
    one = 16   # non-null, 16-byte aligned stand-ins: rejected before any use

    def fwd(R, d, f, fan_out):
        return lib.moe_mlp_fwd(one, d, one, one, one, None, None, 0, 0.0, one, one, one, one, d, one, 0, one, 0, 8,
                               R, d, f, fan_out, 0, 0, None, None, 0, None)
    # a gathered x of 4 GiB or more: T * ldx * 2 bytes
    assert fwd(2 * 600000, 4096, 14336, 2) == -2
    # one expert's matrix of 4 GiB or more
    assert fwd(8192, 65536, 32768, 2) == -2
    # many rows alone are fine: the call gets as far as the workspace check (status -3), i.e. past the size checks
    assert fwd(2 * 200000, 4096, 14336, 2) == -3
    assert lib.moe_mlp_workspace_bytes(400000, 8, 4096, 14336, 16) > 0


def test_fused_layer_rank_limit_is_checked_on_the_host():
    """The fused layer takes an adapter as up to eight chunks of 16 rank columns: rank 128 gets past the shape checks (as
    far as the workspace check), rank 129 is refused with MOE_ERR_UNSUPPORTED before anything is enqueued; the sizes of
    the saved interims and of the workspace grow with the number of chunks."""
    import ctypes
    from moe_distributed_training_amd._lib import lib
    one = 16   # non-null, 16-byte aligned stand-ins: never dereferenced
    lora = (ctypes.c_void_p * 6)(*([one] * 6))
    strides = (ctypes.c_int64 * 18)(*([1] * 18))

    def fwd(rank):
        return lib.moe_mlp_fwd(one, 4096, one, one, one, lora, strides, rank, 1.0, one, one, one, one, 4096, one, 0, one, 0,
                               8, 8192, 4096, 14336, 2, 0, 0, one, None, 0, None)
    assert fwd(128) == -3 and fwd(72) == -3 and fwd(16) == -3
    assert fwd(129) == -2 and fwd(256) == -2
    saved = [lib.moe_mlp_saved_bytes(8192, r) for r in (16, 17, 32, 33, 128)]
    assert saved[1] == saved[2] == 2 * saved[0] and saved[3] == 3 * saved[0] and saved[4] == 8 * saved[0]
    ws = [lib.moe_mlp_workspace_bytes(8192, 8, 4096, 14336, r) for r in (0, 16, 32, 64, 128)]
    assert ws == sorted(ws) and len(set(ws)) == 5


def test_gated_fp16_rows_are_refused_by_the_projection_backward():
    """dY B^T is stored before its gate weight: fp16 with gates, whose range that can pass, is refused with MOE_ERR_UNSUPPORTED before anything is
    enqueued; bf16 with gates and fp16 without get as far as the workspace check."""
    from moe_distributed_training_amd._lib import lib
    one, K, N = 16, 256, 512   # (one: a non-null, 16-byte aligned stand-in, never dereferenced)

    def bwd(dtype, gates):
        return lib.moe_linear_lora_bwd(one, N, 2, gates, 2, one, K, 2, one, K * N, 1, K, one, K * 16, 16, 1, one, 16 * N, N, 1, 16, 1.0, one, K * 16, 16, 1,
                                       one, 16 * N, N, 1, one, K, one, 0, one, 0, 4, 128, K, N, dtype, None, 0, None)
    assert bwd(1, one) == -2
    assert bwd(1, None) == -3 and bwd(0, one) == -3 and bwd(0, None) == -3


def test_the_projection_backward_names_the_sizes_it_refuses():
    """The workspace query is 0 for the sizes that the entry point refuses, so that a caller need not allocate to find out."""
    from moe_distributed_training_amd._lib import lib
    need = lambda K, N, r: lib.moe_linear_lora_bwd_workspace_bytes(128, 4, K, N, r)
    assert all(need(*s) > 0 for s in ((32, 64, 1), (256, 512, 16), (96, 160, 64)))
    assert all(need(*s) == 0 for s in ((256, 512, 65), (256, 512, 0), (48, 64, 16), (64, 48, 16), (64, 32, 16)))


def test_the_mlp_workspace_holds_no_set_of_partials_twice():
    """Rank 16: beside the packed factors, the interims, the column-tile partials of the gate/up and dh launches and three sets of row-tile
    partials of the wider of d and f, everything shares space with the K-split exchange, whose size the query gives for rank 0."""
    from moe_distributed_training_amd._lib import lib
    up = lambda n, m: -(-n // m) * m
    for R, E, d, f in ((8192, 8, 4096, 14336), (32768, 8, 4096, 14336), (16384, 64, 2048, 1024), (1024, 8, 256, 512), (2, 8, 4096, 14336)):
        factors = 3 * 32 * E * (d + f)
        interims = 7 * up(up(R, 32) * 32 + 1024, 256)
        xtp = 3 * (R // 256 + E) * max(d, f) * 64
        columns = 2 * up(f, 256) // 256 * R * 64
        assert lib.moe_mlp_workspace_bytes(R, E, d, f, 16) <= lib.moe_mlp_workspace_bytes(R, E, d, f, 0) + factors + interims + xtp + columns + 4096


def test_the_sum_of_adapter_partials_divides_by_constants(tmp_path):
    """The launch that adds the adapter gradients' partials is a few us of trips to memory: the rows of a partial are constants in every variant of it, and no
    32-bit division by a number known at run time (which starts with v_rcp_iflag_f32) stands before the first load."""
    import shutil
    import subprocess
    import pytest
    if shutil.which("hipcc") is None:
        pytest.skip("no hipcc")
    csrc = os.path.join(ROOT, "moe-distributed-training_amd", "csrc")
    out = str(tmp_path / "lora_kernels.s")
    subprocess.run(["hipcc", "-O3", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-w", "--offload-device-only", "-S",
                    os.path.join(csrc, "lora_kernels.hip"), "-o", out], check=True, timeout=300)
    bodies = dict(re.findall(r"^(\w*xtp_reduce_kernel\w*):[^\n]*\n(.*?)^\s*s_endpgm", open(out).read(), flags=re.S | re.M))
    assert len(bodies) >= 2
    for name, body in bodies.items():
        assert "v_rcp_iflag_f32" not in body, name
