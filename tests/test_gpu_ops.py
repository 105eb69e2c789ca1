"""Operator-level parity of the HIP path (called through the C ABI by the Python mirror of the reference's plugin
surface) against the CPU oracle.  Tolerances: fp32 1e-5 relative to the output scale; bf16 max rel err 1e-2
(fp32 accumulate), the bar the path's specification states."""
import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 2e-5, torch.bfloat16: 1e-2, torch.float16: 2e-3}


from _metrics import rel, rel_per_expert


def check_expert_grads(got, want, tol, what=""):
    """Gradients whose first dimension is the expert: every expert's slice against its own scale (a one-row group must
    meet the bound on its own), max and RMS."""
    mx, rms = rel_per_expert(got, want, with_rms=True)
    assert mx < tol and rms < tol, f"{what}: per-expert max rel err {mx:.4g}, rms rel err {rms:.4g}"


def _tile(R, E, K, N, pair=False, nseg=1):
    """Rows and columns of the output tiles that a launch of these sizes takes."""
    from moe_distributed_training_amd._lib import lib
    return lib.moe_gemm_debug_tile(R, E, K, N, int(pair), nseg)


def _ops():
    from moe_distributed_training_amd.scattermoe_utils.kernels import ops
    return ops


def _routing(oracle, T, E, k, seed=0, skew=False):
    g = torch.Generator().manual_seed(seed)
    logits = torch.randn(T, E, generator=g)
    if skew:
        logits[:, 0] += 3.0
        logits[:, -1] -= 6.0
    idx = torch.topk(logits, k, dim=-1).indices
    sei, ssi = oracle.flatten_and_sort(idx)
    eo = torch.bincount(sei, minlength=E).cumsum(0)
    return idx, sei, ssi, eo


CASES = [
    # dtype, T, E, k, K, N, r
    (torch.float32, 10, 2, 1, 128, 16, 16),      # the reference's own test shape
    (torch.float32, 300, 4, 2, 100, 36, 4),
    (torch.float16, 300, 4, 2, 64, 40, 8),       # fp16 on the matrix cores
    (torch.bfloat16, 300, 4, 2, 72, 40, 8),      # K not a multiple of 64: a partial last K tile, masked loads
    (torch.float16, 700, 8, 2, 200, 264, 16),    # fp16, three whole K tiles and a partial one, N tail, adapters
    (torch.bfloat16, 500, 4, 2, 1096, 512, 24),  # split K with a partial last tile, two adapter slabs
    (torch.bfloat16, 300, 4, 2, 40, 64, 8),      # K below one K tile -> generic kernels
    (torch.bfloat16, 1000, 8, 2, 256, 512, 16),
    (torch.bfloat16, 1500, 8, 2, 512, 264, 16),  # N tail inside a 256-wide tile
    (torch.bfloat16, 700, 3, 2, 1024, 256, 4),   # rank < 16 zero padded
    (torch.bfloat16, 2500, 8, 2, 128, 1280, 16),
    (torch.bfloat16, 600, 4, 2, 2048, 512, 16),  # few tiles, deep K: every tile is cut 4 ways along K
    (torch.bfloat16, 400, 4, 2, 256, 512, 32),   # rank above 16: the adapter enters as two 16-wide slabs
    (torch.bfloat16, 400, 4, 2, 256, 512, 64),   # four slabs in two MFMA steps
    (torch.bfloat16, 400, 4, 2, 256, 512, 40),   # three slabs, the last one partly filled
    (torch.bfloat16, 400, 4, 2, 256, 512, 96),   # a rank above 64: six slabs at a fixed stride, two per step in a loop
    (torch.float16, 400, 4, 2, 264, 256, 136),   # nine slabs (the last half empty), fp16, and a partial last K tile
    (torch.bfloat16, 1200, 96, 4, 256, 512, 16), # more than 64 experts (group lookup in blocks of 64), top-4, every tile ragged
    (torch.bfloat16, 500, 4, 2, 64, 512, 16),    # a single K tile: the adapter slabs' LDS image is requested before the loop
    (torch.bfloat16, 500, 4, 2, 192, 300, 16),   # three K tiles: ... by the first trip through the loop
]
# The cases above are small and take 128 x 128 tiles where their K is a multiple of 64; the same forms in the 256 x 256 tiles of larger launches
LARGE_TILE_CASES = [
    (torch.bfloat16, 1500, 8, 2, 256, 2048, 16),
    (torch.bfloat16, 1500, 8, 2, 256, 2048, 32),  # two slabs
    (torch.bfloat16, 1500, 8, 2, 256, 2048, 40),  # three, the last one partly filled
    (torch.float16, 1500, 8, 2, 256, 2048, 64),   # four
    (torch.bfloat16, 1100, 4, 2, 2048, 1024, 16), # every tile cut along K
    (torch.bfloat16, 1500, 8, 2, 64, 2048, 16),   # a single K tile
    (torch.bfloat16, 1500, 8, 2, 192, 2056, 16),  # three, and an N tail
]


@pytest.mark.parametrize("layout", ["k_contiguous", "n_contiguous"])
@pytest.mark.parametrize("dtype,T,E,k,K,N,r", CASES + LARGE_TILE_CASES)
def test_scatter2scatter_all_row_mappings(dev, oracle, layout, dtype, T, E, k, K, N, r):
    ops = _ops()
    torch.manual_seed(1)
    _, sei, ssi, eo = _routing(oracle, T, E, k, skew=True)
    W = (torch.randn(E, N, K) * 0.05).to(dtype).permute(0, 2, 1) if layout == "k_contiguous" else (torch.randn(E, K, N) * 0.05).to(dtype)
    A = (torch.randn(E, K, r) * 0.05).to(dtype)
    B = (torch.randn(E, r, N) * 0.05).to(dtype)
    seid, ssid = sei.to(dev), ssi.int().to(dev)            # mixed index widths on purpose
    # which kernel a shape takes: 2-byte types with K >= 64 and K, N multiples of 8 run on the matrix cores (one grouped
    # GEMM launch per call), everything else on the generic kernels
    from moe_distributed_training_amd._lib import lib
    on_matrix_cores = dtype != torch.float32 and K >= 64 and K % 8 == 0 and N % 8 == 0
    if (dtype, T, E, k, K, N, r) in LARGE_TILE_CASES:
        assert _tile(T * k, E, K, N) == 256
    for xg, yg in [(False, True), (False, False), (True, False), (True, True)]:
        X = torch.randn(T * k if xg else T, K).to(dtype)
        kk = 1 if xg else k
        s_in = ssi if not xg else ssi
        n0 = lib.moe_gemm_debug_launch_count()
        y = ops.scatter2scatter_lora(X.to(dev), W.to(dev), A.to(dev), B.to(dev), 32.0, seid, ssid, kk, None, xg, yg)
        assert lib.moe_gemm_debug_launch_count() - n0 == int(on_matrix_cores)
        yo = oracle.scatter2scatter_lora(X, W, A, B, 32.0, sei, s_in, kk, None, xg, yg)
        assert rel(y, yo) < TOL[dtype], (xg, yg)
        y2 = ops.scatter2scatter(X.to(dev), W.to(dev), seid, ssid, kk, None, xg, yg)
        assert lib.moe_gemm_debug_launch_count() - n0 == 2 * int(on_matrix_cores)
        yo2 = oracle.scatter2scatter_lora(X, W, None, None, 0.0, sei, s_in, kk, None, xg, yg)
        assert rel(y2, yo2) < TOL[dtype], (xg, yg)


@pytest.mark.parametrize("T,E,k,K,N,layout,tile", [(600, 4, 2, 2048, 512, "k_contiguous", 128), (600, 4, 2, 2048, 512, "n_contiguous", 128),
                                                   (1100, 4, 2, 2048, 1024, "k_contiguous", 256), (4096, 8, 2, 14336, 4096, "n_contiguous", 256)])
def test_k_split_exchange_is_stable_over_many_launches(dev, oracle, T, E, k, K, N, layout, tile):
    """Tiles of the last, partial round are cut 2 or 4 ways along K; the parts exchange fp32 partials through memory
    that crosses the XCDs' separate L2 caches and a counter.  A stale read there would be a silent, intermittent wrong
    sum: 2000 launches of the same problem (small ones where every tile is split, in tiles of either size, and the h W2 product at
    the Mixtral shape) must all be bitwise equal to the first, which itself meets the oracle; stops at the first mismatch."""
    ops = _ops()
    torch.manual_seed(21)
    _, sei, ssi, eo = _routing(oracle, T, E, k, seed=21)
    L = T * k
    g = torch.Generator(device=dev).manual_seed(22)
    X = torch.randn(L, K, generator=g, device=dev).bfloat16()
    W = (torch.randn(E, N, K, generator=g, device=dev) * 0.05).bfloat16().permute(0, 2, 1) if layout == "k_contiguous" else \
        (torch.randn(E, K, N, generator=g, device=dev) * 0.05).bfloat16()
    seid, ssid = sei.to(dev), ssi.int().to(dev)
    assert _tile(L, E, K, N) == tile
    plan, _ = _plan(dev, torch.bincount(sei, minlength=E).tolist(), K, N, False)
    assert (plan[:, 0] == 1).any() and (plan[plan[:, 0] == 1][:, 6] > 1).any(), "the case must have K-split tiles"
    first = ops.scatter2scatter(X, W, seid, ssid, 1, None, True, True)
    if L * K * N <= 2e10:
        ref = oracle.scatter2scatter_lora(X.float().cpu(), W.float().cpu(), None, None, 0.0, sei, ssi, 1, None, True, True)
        assert rel(first, ref) < 1e-2
    out = torch.empty_like(first)
    bad = torch.zeros((), dtype=torch.int32, device=dev)
    launches, check_every = 2000, 100
    for i in range(launches):
        ops.scatter2scatter(X, W, seid, ssid, 1, None, True, True, out=out)
        bad += (out != first).any().int()
        if (i + 1) % check_every == 0:
            assert int(bad.item()) == 0, f"a launch among {i + 2 - check_every}..{i + 1} differs from the first"


@pytest.mark.slow
@pytest.mark.parametrize("case", ["grouped_out_above_2GiB", "scattered_out_above_2GiB", "grouped_in_above_4GiB"])
def test_scatter2scatter_beyond_32_bit_spans(dev, case):
    """Tensors larger than a 32-bit byte offset reaches: a grouped output above 2 GiB (tiles addressed from their own
    first row), a scattered output above 2 GiB (64-bit row addresses) and a grouped input above 4 GiB.  Rows from the
    first tile, the last tile and around the 2 / 4 GiB marks against per-row fp32 products."""
    ops = _ops()
    g = torch.Generator(device=dev).manual_seed(31)
    E = 4
    if case == "grouped_in_above_4GiB":
        R, K, N = 140000, 16384, 64
    else:
        R, K, N = 70000, 64, 16384
    counts = [R // 2 - 777, 0, R // 4 + 500, R - (R // 2 - 777) - (R // 4 + 500)]
    eo = torch.tensor(counts).cumsum(0)
    sei = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).to(dev)
    scattered = case == "scattered_out_above_2GiB"
    ssi = (torch.randperm(R, generator=torch.Generator().manual_seed(32)) if scattered else torch.arange(R)).to(dev)
    X = torch.randn(R, K, generator=g, device=dev).bfloat16()
    W = (torch.randn(E, K, N, generator=g, device=dev) * 0.05).bfloat16()
    assert max(X.numel(), R * N) * 2 > (1 << 31)
    y = ops.scatter2scatter(X, W, sei, ssi, 1, None, True, not scattered)
    torch.cuda.synchronize()
    mark = (1 << 31) // (2 * N) if case != "grouped_in_above_4GiB" else (1 << 32) // (2 * K)
    rows = sorted(set(list(range(0, 300)) + list(range(R - 300, R)) + list(range(mark - 300, mark + 300)) +
                      [int(v) for v in eo.tolist() if 0 < v < R] + [int(v) - 1 for v in eo.tolist() if v > 0]))
    m = torch.tensor(rows, device=dev)
    e_of = sei[m]
    ref = torch.bmm(X[m].float().unsqueeze(1), W.float()[e_of]).squeeze(1)
    got = y[ssi[m] if scattered else m].float()
    assert float((got - ref).abs().max() / ref.abs().max()) < 1e-2
    if scattered:   # every output row was written exactly once: a permutation of the grouped result
        yg = ops.scatter2scatter(X, W, sei, ssi, 1, None, True, True)
        assert torch.equal(y[ssi], yg)


def test_scatter2scatter_out_argument_and_empty(dev, oracle):
    ops = _ops()
    torch.manual_seed(2)
    T, E, k, K, N = 64, 4, 2, 64, 64
    _, sei, ssi, eo = _routing(oracle, T, E, k)
    X = torch.randn(T, K).bfloat16(); W = (torch.randn(E, K, N) * 0.1).bfloat16()
    out = torch.zeros(T * k, N, dtype=torch.bfloat16, device=dev)
    y = ops.scatter2scatter(X.to(dev), W.to(dev), sei.to(dev), ssi.to(dev), k, None, False, True, out=out)
    assert y.data_ptr() == out.data_ptr()
    assert rel(out, oracle.scatter2scatter_lora(X, W, None, None, 0, sei, ssi, k, None, False, True)) < 1e-2
    with pytest.raises(AssertionError):
        ops.scatter2scatter(X.to(dev), W.to(dev), sei.to(dev), ssi.to(dev), 1, None, False, True)   # rows(X)*k mismatch
    e = torch.empty(0, dtype=torch.int64, device=dev)
    y0 = ops.scatter2scatter(X[:0].to(dev), W.to(dev), e, e, k)
    assert y0.shape == (0, N)


@pytest.mark.parametrize("counts,K,N", [([17, 0, 1, 16, 15, 300], 64, 256), ([5, 130, 33], 63, 513), ([16] * 9, 65, 449), ([700, 324], 1, 80), ([700, 324], 31, 200), ([40, 60], 130, 1000),
                                        ([17, 0, 1, 16, 15, 300] * 3, 64, 512), ([50, 1030, 333], 63, 513), ([16] * 36, 65, 449), ([4700, 1324], 1, 80), ([1700, 324], 31, 200), ([40, 160], 130, 1000)])
@pytest.mark.parametrize("layout", ["k", "n", "wide"])
@pytest.mark.parametrize("gathered", [False, True])
def test_fp32_products_on_the_matrix_cores(dev, counts, K, N, layout, gathered):
    """fp32 products without adapters, edges of their 16-row, 64-column and 64-k tiles, weights contiguous along k or n or along neither, rows grouped or
    gathered and scattered, against 64 bits; the same edges in launches of few tiles (the vector kernel) and of more.  Bound: a result is a sum of K products, each rounding at most 2^-24 of the sum of their magnitudes."""
    ops = _ops()
    g = torch.Generator().manual_seed(K + N)
    E, R = len(counts), sum(counts)
    X = torch.randn(R, K, generator=g)
    W = torch.randn(E, K, N, generator=g)
    order = torch.randperm(R, generator=g) if gathered else torch.arange(R)
    sei = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    Wd = W.to(dev)
    if layout == "k":
        Wd = Wd.transpose(1, 2).contiguous().transpose(1, 2)
    elif layout == "wide":
        Wd = torch.empty(E, K, 2 * N, device=dev)[:, :, ::2].copy_(Wd)
    y = ops.scatter2scatter(X.to(dev), Wd, sei.to(dev), order.to(dev), 1, None, not gathered, not gathered).cpu().double()
    rows = X[order].double() if gathered else X.double()
    ref = torch.cat([rows[sei == e] @ W[e].double() for e in range(E)])
    mag = torch.cat([rows[sei == e].abs() @ W[e].double().abs() for e in range(E)])
    got = y[order] if gathered else y
    assert bool(((got - ref).abs() <= K * 2.0 ** -24 * mag + 1e-30).all())


@pytest.mark.parametrize("counts,K,N,cores", [
    ([128] * 4, 256, 128, False), ([1] * 8, 512, 512, False), ([1] * 8, 256, 1024, False), ([512] * 4, 64, 80, False), ([512] * 4, 512, 48, False), ([256] * 2, 40, 384, False),
    ([128] * 4, 128, 256, True), ([256] * 2, 64, 384, True), ([1] * 8, 128, 2048, True), ([256] * 2, 40, 512, True), ([2048] * 4, 64, 40, True)])
@pytest.mark.parametrize("pair", [False, True])
def test_which_fp32_products_run_on_the_matrix_cores(dev, counts, K, N, cores, pair):
    """Launches of few tiles are the vector kernel's, which is the faster one there (by up to a quarter), for one product and for gate and up.  The vector kernel adds along k whatever N is, and
    16 columns by themselves are always its own: the bits tell which kernel a launch took."""
    from moe_distributed_training_amd._lib import lib, check, ptr, stream_ptr
    ncu = torch.cuda.get_device_properties(dev).multi_processor_count
    if ncu != 256:
        pytest.skip("the sizes are those of 256 compute units")
    g = torch.Generator().manual_seed(K + N)
    E, R = len(counts), sum(counts)
    X = torch.randn(R, K, generator=g).to(dev)
    W, U = (torch.randn(E, K, N, generator=g).to(dev) for _ in range(2))
    eo, pos = torch.tensor(counts).cumsum(0).int().to(dev), torch.arange(R, dtype=torch.int32, device=dev)
    ops = _ops()
    sei = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).int().to(dev)

    def product(w, u):
        if not pair:
            return ops.scatter2scatter(X, w, sei, pos, 1, None, True, True)
        y = torch.empty(R, w.size(2), device=dev)
        check(lib.moe_swiglu_pair(ptr(X), K, 1, ptr(w), ptr(u), w.stride(0), w.stride(1), 1, ptr(y), y.size(1), ptr(pos), 0, ptr(eo), 0, E, R, K, w.size(2), 1, 2, stream_ptr(dev)), "pair")
        return y
    pieces = torch.cat([product(W[:, :, n:n + 16], U[:, :, n:n + 16]) for n in range(0, N, 16)], 1)
    assert torch.equal(product(W, U), pieces) is not cores


@pytest.mark.parametrize("counts,K,N", [
    ([301, 0, 77, 1, 513], 256, 512),        # ragged groups: empty, one row, not a multiple of the 64-row step
    ([64, 128, 192], 512, 256),              # whole steps only
    ([130, 5, 0, 260], 264, 136),            # K and N not multiples of the 256 tile: edge columns are masked
    ([1000, 3000], 768, 2304),               # several panels of n tiles, long contraction
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_group_bwd_w_matrix_cores(dev, oracle, counts, K, N, dtype):
    """bf16 / fp16 DW[e] = X_e^T DY_e (scattermoe group_bwd_W, full fine-tuning) against the fp32 per-expert matmul; rows of
    the next group must not leak into a group's last, partial contraction step, an empty group gives zeros."""
    ops = _ops()
    torch.manual_seed(11)
    E = len(counts)
    eo = torch.tensor(counts).cumsum(0)
    R = int(eo[-1])
    X = torch.randn(R, K).to(dtype); DY = (torch.randn(R, N) * 0.25).to(dtype)
    ref = oracle.group_bwd_W(DY, X, eo, E)
    for offs in (eo.to(dev), eo.int().to(dev)):
        dW = ops.group_bwd_W(DY.to(dev), X.to(dev), offs, E)
        assert dW.shape == (E, K, N) and dW.dtype == dtype
        for e in range(E):
            if counts[e] == 0:
                assert float(dW[e].abs().max()) == 0.0
            else:
                assert rel(dW[e], ref[e]) < TOL[dtype]
    if dtype != torch.bfloat16:
        return
    # row-strided operands (column slices of wider buffers) take the same kernel
    Xw = torch.randn(R, K + 64).bfloat16().to(dev); DYw = torch.randn(R, N + 8).bfloat16().to(dev)
    dW = ops.group_bwd_W(DYw[:, 8:], Xw[:, 64:], eo.to(dev), E)
    check_expert_grads(dW, oracle.group_bwd_W(DYw[:, 8:].cpu(), Xw[:, 64:].cpu(), eo, E), TOL[torch.bfloat16], "dW strided")


def test_group_bwd_w_mixtral_shape(dev, oracle):
    """Full size of one Mixtral projection (R=8192 rows in 8 ragged groups, K=4096, N=14336): every expert's matrix
    against the fp32 per-expert matmul on the host."""
    ops = _ops()
    g = torch.Generator(device=dev).manual_seed(5)
    counts = [1100, 950, 1030, 1200, 900, 1012, 1000, 1000]
    eo = torch.tensor(counts).cumsum(0)
    X = torch.randn(8192, 4096, generator=g, device=dev).bfloat16()
    DY = torch.randn(8192, 14336, generator=g, device=dev).bfloat16()
    dW = ops.group_bwd_W(DY, X, eo.to(dev), 8)
    torch.cuda.synchronize()
    torch.set_num_threads(16)
    Xc, DYc = X.float().cpu(), DY.float().cpu()
    start = 0
    for e, c in enumerate(counts):
        ref = Xc[start:start + c].T @ DYc[start:start + c]
        assert rel(dW[e], ref) < TOL[torch.bfloat16], f"expert {e}"
        start += c


@pytest.mark.parametrize("dtype,K,N,r", [(torch.float32, 150, 140, 4), (torch.bfloat16, 256, 512, 16), (torch.bfloat16, 256, 512, 64),
                                         (torch.bfloat16, 4096, 1024, 16), (torch.bfloat16, 96, 160, 8),
                                         (torch.float16, 130, 70, 16), (torch.float16, 256, 512, 16), (torch.float16, 512, 288, 48)])
def test_group_bwd_ab_full_reduction(dev, oracle, dtype, K, N, r):
    """K and N above 128 on purpose: every N tile must contribute to dA and every K tile to dB."""
    ops = _ops()
    torch.manual_seed(3)
    E = 5
    counts = torch.tensor([301, 0, 77, 1, 513])
    eo = counts.cumsum(0)
    R = int(eo[-1])
    X = torch.randn(R, K).to(dtype); DY = torch.randn(R, N).to(dtype)
    A = (torch.randn(E, K, r) * 0.1).to(dtype); B = (torch.randn(E, r, N) * 0.1).to(dtype)
    dA, dB = ops.group_bwd_AB(DY.to(dev), X.to(dev), A.to(dev), B.to(dev), 2.0, eo.to(dev), E)
    dAo, dBo = oracle.group_bwd_AB(DY, X, A, B, 2.0, eo, E)
    assert dA.shape == (E, K, r) and dB.shape == (E, r, N) and dA.dtype == dtype
    check_expert_grads(dA, dAo, TOL[dtype] * 1.5, "dA"); check_expert_grads(dB, dBo, TOL[dtype] * 1.5, "dB")
    assert float(dA[1].abs().max()) == 0.0 and float(dB[1].abs().max()) == 0.0
    dW = ops.group_bwd_W(DY.to(dev), X.to(dev), eo.int().to(dev), E)
    check_expert_grads(dW, oracle.group_bwd_W(DY, X, eo, E), TOL[dtype] * 1.5, "dW")
    # strided adapter views (the w2 arrangement of the reference: both factors permuted)
    A2 = (torch.randn(E, r, K) * 0.1).to(dtype).permute(0, 2, 1); B2 = (torch.randn(E, N, r) * 0.1).to(dtype).permute(0, 2, 1)
    dA2, dB2 = ops.group_bwd_AB(DY.to(dev), X.to(dev), A2.to(dev), B2.to(dev), 0.5, eo.to(dev), E)
    dAo2, dBo2 = oracle.group_bwd_AB(DY, X, A2, B2, 0.5, eo, E)
    check_expert_grads(dA2, dAo2, TOL[dtype] * 1.5, "dA strided"); check_expert_grads(dB2, dBo2, TOL[dtype] * 1.5, "dB strided")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_group_and_combine(dev, oracle, dtype):
    ops = _ops()
    torch.manual_seed(4)
    T, E, k, N = 257, 6, 2, 200
    _, sei, ssi, eo = _routing(oracle, T, E, k)
    src = torch.randn(T, N).to(dtype); coeff = torch.rand(T * k).to(dtype)
    g = ops.group(src.to(dev), ssi.to(dev), coeff=coeff.to(dev), fan_out=k)
    assert rel(g, oracle.group(src.float(), ssi, coeff.float(), k)) < TOL[dtype]
    g1 = ops.group(src.to(dev), ssi.to(dev), fan_out=k)
    assert torch.equal(g1.cpu(), src[ssi // k])
    yg = torch.randn(T * k, N).to(dtype); w = torch.rand(T, k)
    inv = torch.empty(T * k, dtype=torch.int32); inv[ssi] = torch.arange(T * k, dtype=torch.int32)
    out = ops.combine(yg.to(dev), w.to(dev), inv=inv.to(dev))
    assert rel(out, oracle.combine(yg.float(), ssi, w, T, k)) < TOL[dtype]
    dout = torch.randn(T, N).to(dtype)
    dg = ops.combine_dgates(yg.to(dev), dout.to(dev), k, torch.float32, inv=inv.to(dev))
    ref = (yg.float()[inv.long()].view(T, k, N) * dout.float()[:, None, :]).sum(-1)
    assert rel(dg, ref) < TOL[dtype]


def _run_parallel_linear(dev, oracle, dtype, T, E, k, K, N, r, gates, gin, gout, lora=True, seed=5):
    import moe_distributed_training_amd as moe
    torch.manual_seed(seed)
    _, sei, ssi, eo = _routing(oracle, T, E, k, seed)
    L = T * k
    X = torch.randn(L if gin else T, K).to(dtype)
    W = (torch.randn(E, N, K) * 0.05).to(dtype).permute(0, 2, 1)
    A = (torch.randn(E, K, r) * 0.05).to(dtype); B = (torch.randn(E, r, N) * 0.05).to(dtype)
    G = torch.rand(T, k).to(dtype) if gates else None
    kk = 1 if gin else k
    rows_out = T if gates else L
    dY = torch.randn(rows_out, N).to(dtype)
    f32 = lambda t: None if t is None else t.detach().float().clone().requires_grad_(True)
    Xo, Wo, Ao, Bo, Go = f32(X), f32(W), f32(A), f32(B), f32(G)
    yo = oracle.parallel_linear_lora(Xo, Wo, Ao if lora else None, Bo if lora else None, r, 32.0, kk, sei, ssi, None, eo,
                                     Go, gin, gout)
    yo.backward(dY.float())
    d = lambda t: None if t is None else t.detach().to(dev).requires_grad_(True)
    Xd, Wd, Ad, Bd, Gd = d(X), d(W), d(A), d(B), d(G)
    pb, eod = moe.padded_block_indices(sei.to(dev), E)
    if lora:
        y = moe.parallel_linear_lora(Xd, Wd, Ad, Bd, r, 32.0, kk, sei.to(dev), ssi.to(dev), pb, eod, Gd, gin, gout)
    else:
        y = moe.parallel_linear(Xd, Wd, kk, sei.to(dev), ssi.to(dev), pb, eod, Gd, gin, gout)
    y.backward(dY.to(dev))
    tol = TOL[dtype] * 1.5
    assert rel(y, yo) < tol
    assert rel(Xd.grad, Xo.grad) < tol
    if lora:
        check_expert_grads(Ad.grad, Ao.grad, tol, "dA"); check_expert_grads(Bd.grad, Bo.grad, tol, "dB")
        assert Wd.grad is None                                   # base weights are frozen on the LoRA path
    else:
        check_expert_grads(Wd.grad, Wo.grad, tol, "dW")
    if gates:
        assert rel(Gd.grad, Go.grad) < tol


@pytest.mark.parametrize("dtype,K,N,r", [(torch.float32, 128, 16, 16), (torch.bfloat16, 256, 384, 16), (torch.bfloat16, 200, 136, 16),
                                         (torch.bfloat16, 256, 384, 32), (torch.float16, 256, 384, 16)])
@pytest.mark.parametrize("gates,gin,gout", [(False, False, True), (False, True, False), (True, False, False), (False, False, False), (False, True, True)])
def test_parallel_linear_lora_autograd(dev, oracle, dtype, K, N, r, gates, gin, gout):
    _run_parallel_linear(dev, oracle, dtype, 333, 4, 2, K, N, r, gates, gin, gout)


@pytest.mark.parametrize("gates,gin,gout", [(False, False, True), (True, False, False), (False, True, False)])
def test_parallel_linear_plain_autograd_with_dw(dev, oracle, gates, gin, gout):
    _run_parallel_linear(dev, oracle, torch.bfloat16, 333, 4, 2, 256, 128, 16, gates, gin, gout, lora=False)
    _run_parallel_linear(dev, oracle, torch.float32, 100, 3, 2, 50, 30, 16, gates, gin, gout, lora=False)


def test_reference_test_case(dev, oracle):
    """tests/test_scattermoe.py of the reference: E=2, 128 -> 16, r=16, alpha=32, 10 rows, k=1, scattered in, grouped
    out, loss = out.norm(); output and dB compared at atol=1e-2 (here also dA and dX)."""
    import moe_distributed_training_amd as moe
    torch.manual_seed(42)
    X = torch.randn(10, 128)
    sei = torch.tensor([0, 0, 0, 0, 1, 1, 1, 1, 1, 1]); ssi = torch.tensor([4, 6, 8, 9, 0, 1, 2, 3, 5, 7])
    lin = [torch.nn.Linear(128, 16, bias=False) for _ in range(2)]
    W = torch.stack([l.weight.detach().T for l in lin])
    A = torch.randn(2, 128, 16) * 0.02; B = torch.randn(2, 16, 16) * 0.02
    Ao, Bo, Xo = A.clone().requires_grad_(True), B.clone().requires_grad_(True), X.clone().requires_grad_(True)
    out = torch.cat([Xo[ssi[sei == i]] @ (W[i] + 2.0 * Ao[i] @ Bo[i]) for i in range(2)])     # ExpertModel loop + LoRA
    out.norm().backward()
    Xd, Ad, Bd = X.to(dev).requires_grad_(True), A.to(dev).requires_grad_(True), B.to(dev).requires_grad_(True)
    pb, eo = moe.padded_block_indices(sei.to(dev), 2)
    out2 = moe.parallel_linear_lora(Xd, W.to(dev), Ad, Bd, 16, 32, 1, sei.to(dev), ssi.to(dev), pb, eo,
                                    grouped_in=False, grouped_out=True)
    out2.norm().backward()
    assert torch.allclose(out, out2.cpu(), atol=1e-2)
    assert torch.allclose(Bo.grad, Bd.grad.cpu(), atol=1e-2) and torch.allclose(Ao.grad, Ad.grad.cpu(), atol=1e-2)
    assert torch.allclose(out, out2.cpu(), atol=1e-5) and torch.allclose(Bo.grad, Bd.grad.cpu(), atol=1e-5)
    assert torch.allclose(Xo.grad, Xd.grad.cpu(), atol=1e-5)


def test_parallel_experts_module(dev, oracle):
    import moe_distributed_training_amd as moe
    torch.manual_seed(6)
    T, E, k, K, N = 128, 4, 2, 64, 128
    m = moe.ParallelExperts(E, K, N, device=dev, dtype=torch.bfloat16)
    assert m.weight.shape == (E, N, K)
    _, sei, ssi, eo = _routing(oracle, T, E, k)
    X = torch.randn(T, K).bfloat16()
    y = m(X.to(dev), k, sei.to(dev), ssi.to(dev), None, eo.to(dev), grouped_out=True)
    yo = oracle.scatter2scatter_lora(X, m.weight.detach().cpu().permute(0, 2, 1), None, None, 0, sei, ssi, k, None, False, True)
    assert rel(y, yo) < 1e-2


def _plan(dev, counts, K, N, pair, nseg=1, tile=None):
    from moe_distributed_training_amd._lib import lib, check, ptr, stream_ptr
    E = len(counts)
    R = int(sum(counts))
    eo = torch.tensor(counts, dtype=torch.int64).cumsum(0).to(dev)
    tile = tile or _tile(R, E, K, N, pair, nseg)
    blocks = lib.moe_gemm_debug_tile_plan_blocks(tile, R, E, N, int(pair))
    out = torch.full((blocks, 9), -7, dtype=torch.int32, device=dev)
    check(lib.moe_gemm_debug_tile_plan(tile, ptr(eo), 1, E, R, K, N, int(pair), nseg, ptr(out), stream_ptr(dev)), "moe_gemm_debug_tile_plan")
    return out.cpu().numpy(), blocks


@pytest.mark.parametrize("tile", [256, 128])
@pytest.mark.parametrize("case", range(32))
def test_grouped_gemm_tile_plan_covers_every_tile_once(dev, case, tile):
    """The work items the grouped GEMM's workgroups decode for themselves, for seeded group sizes (even, ragged, skewed,
    empty groups, few and many rounds of tiles, both tile sizes and widths, more experts than one wave looks up at once): the rows of a
    group are cut into as many tiles as it needs, without a gap, at 16-row blocks and to within one block evenly; every output
    tile appears exactly once, either whole or as K parts 0..n-1 with consecutive exchange slots and one counter, and slots and
    counters are unique and within the exchange area's size."""
    import random
    rng = random.Random(500 + case)
    E = rng.choice([1, 2, 3, 8, 8, 8, 17, 64]) if case < 24 else rng.choice([65, 96, 130])
    kind = rng.choice(["even", "ragged", "skewed", "tiny"])
    R = rng.choice([300, 2000, 8192, 8192, 20000])
    if kind == "even":
        counts = [R // E] * E
    elif kind == "ragged":
        counts = [max(0, int(R / E * (1 + 0.15 * rng.uniform(-1, 1)))) for _ in range(E)]
    elif kind == "skewed":
        w = [1.0 / (i + 1) ** 1.2 for i in range(E)]
        counts = [int(R * x / sum(w)) for x in w]
        rng.shuffle(counts)
    else:
        counts = [rng.choice([0, 0, 1, 5, 40, 130, 257]) for _ in range(E)]
    if sum(counts) == 0:
        counts[0] = 3
    if case >= 24:   # groups of several tiles among the first and the last experts of each 64
        for e, c in ((0, 272), (63, 1060), (64, 257), (E - 1, 600)):
            counts[e] = c
    K = rng.choice([512, 4096, 14336])
    N = rng.choice([256, 4096, 14336, 1000])
    pair = rng.choice([False, True])
    nseg = 1 if pair else rng.choice([1, 2])
    plan, blocks = _plan(dev, counts, K, N, pair, nseg, tile)
    ncu = torch.cuda.get_device_properties(dev).multi_processor_count // 8 * 8
    bn = tile // 2 if pair else tile
    ntn = (N + bn - 1) // bn
    tiles_ub = (sum(counts) // tile + E) * ((N + tile - 1) // tile)
    slots_cap = min(4 * tiles_ub, 256 // tile * ncu)   # one round of workgroups; the counters, one per compute unit, are half as many with small tiles
    seen = {}
    for b in range(blocks):
        valid, e, ntile, r0, r1, part, nparts, slot, counter = (int(v) for v in plan[b])
        assert valid in (0, 1), f"block {b} wrote nothing"
        if not valid:
            continue
        key = (e, ntile, r0, r1)
        assert nparts in (1, 2, 4) and 0 <= part < nparts
        seen.setdefault(key, []).append((part, nparts, slot, counter))
    rows = {}
    for e, ntile, r0, r1 in seen:
        rows.setdefault((e, ntile), []).append((r0, r1))
    assert set(rows) == {(e, ntile) for e, c in enumerate(counts) if c for ntile in range(ntn)}, case
    ends = [sum(counts[:e + 1]) for e in range(E)]
    for (e, ntile), cut in rows.items():
        cut.sort()
        blocks_of = [(r1 - r0 + 15) // 16 for r0, r1 in cut]
        assert len(cut) == (counts[e] + tile - 1) // tile and cut[0][0] == ends[e] - counts[e] and cut[-1][1] == ends[e], (case, e, cut)
        assert all(a[1] == b[0] and (a[1] - a[0]) % 16 == 0 for a, b in zip(cut, cut[1:])), (case, e, cut)
        assert max(blocks_of) <= tile // 16 and max(blocks_of) - min(blocks_of) <= 1, (case, e, cut)
    used_slots, used_counters = set(), set()
    for key, items in seen.items():
        nparts = items[0][1]
        assert len(items) == nparts and sorted(i[0] for i in items) == list(range(nparts)), (case, key, items)
        if nparts > 1:
            assert max_split_ok(pair), "the pair kernel never splits"
            first = min(i[2] for i in items)
            assert all(i[2] == first + i[0] and i[1] == nparts and i[3] == items[0][3] for i in items), (case, key, items)
            for i in items:
                assert 0 <= i[2] < slots_cap and i[2] not in used_slots
                used_slots.add(i[2])
            assert 0 <= items[0][3] < ncu and items[0][3] not in used_counters
            used_counters.add(items[0][3])


def max_split_ok(pair):
    return not pair



@pytest.mark.parametrize("counts", [[257, 272, 273, 1], [511, 512, 513, 15], [769, 16, 1025, 0], [144, 145, 287, 31]])
@pytest.mark.parametrize("layout", ["k_contiguous", "n_contiguous"])
@pytest.mark.parametrize("N,tile", [(320, 128), (8192, 256)])
def test_grouped_gemm_rows_dealt_evenly_to_tiles(dev, oracle, counts, layout, N, tile):
    """Groups of one block more or less than a whole number of tiles of either size: every row exactly once, whatever tile it falls into."""
    ops = _ops()
    torch.manual_seed(21)
    E, K = len(counts), 512
    R = sum(counts)
    assert _tile(R, E, K, N) == tile
    sei = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    ssi = torch.randperm(R, generator=torch.Generator().manual_seed(2))
    X, W = torch.randn(R, K).bfloat16(), (torch.randn(E, K, N) * 0.05).bfloat16()
    Wd = W.permute(0, 2, 1).contiguous().to(dev).permute(0, 2, 1) if layout == "k_contiguous" else W.to(dev)
    y = ops.scatter2scatter(X.to(dev), Wd, sei.to(dev), ssi.to(dev), 1)
    ref = oracle.scatter2scatter_lora(X, W, None, None, 0, sei, ssi, 1)
    # one bf16 rounding of fp32 sums: half an ulp, 2^-9 of the value, and the sum's own error far below it
    assert float((y.float().cpu() - ref).abs().max()) <= 2.0 ** -8 * float(ref.abs().max())


@pytest.mark.parametrize("E", [65, 130])
def test_grouped_gemm_many_experts_with_several_tiles(dev, oracle, E):
    """Groups of several row tiles among the first and last experts of each 64 that a wave looks up at once."""
    ops = _ops()
    torch.manual_seed(E)
    counts = [3 * (e % 3) for e in range(E)]
    for e, c in ((0, 272), (63, 530), (64, 257), (E - 1, 600)):
        counts[e] = c
    K, N = 128, 320
    sei = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    ssi = torch.randperm(len(sei), generator=torch.Generator().manual_seed(4))
    X, W = torch.randn(len(sei), K).bfloat16(), (torch.randn(E, K, N) * 0.05).bfloat16()
    y = ops.scatter2scatter(X.to(dev), W.to(dev), sei.to(dev), ssi.to(dev), 1)
    ref = oracle.scatter2scatter_lora(X, W, None, None, 0, sei, ssi, 1)
    # one bf16 rounding of fp32 sums: half an ulp, 2^-9 of the value, and the sum's own error far below it
    assert float((y.float().cpu() - ref).abs().max()) <= 2.0 ** -8 * float(ref.abs().max())


@pytest.mark.parametrize("rows", [257, 272, 300, 513, 544])
@pytest.mark.parametrize("layout", ["k_contiguous", "n_contiguous"])
def test_grouped_gemm_tiles_of_a_group_walk_the_same_way(dev, rows, layout):
    """Equal rows of a group have equal bits whichever of its row tiles they fall into: tiles that share their weights take them in one
    order (a tile of half the row blocks among them: 257..272 rows are 9 and 8 blocks)."""
    ops = _ops()
    torch.manual_seed(24)
    E, K, N = 3, 512, 4096
    sei = torch.repeat_interleave(torch.arange(E), torch.tensor([rows, 5, rows])).to(dev)
    ssi = torch.arange(len(sei), device=dev)
    X = torch.randn(1, K, device=dev, dtype=torch.float16).expand(len(sei), K).contiguous()
    W = torch.randn(E, K, N, device=dev, dtype=torch.float16)
    if layout == "k_contiguous":
        W = W.permute(0, 2, 1).contiguous().permute(0, 2, 1)
    y = ops.scatter2scatter(X, W, sei, ssi, 1)
    for e in (0, 2):
        group = y[sei == e]
        assert torch.equal(group, group[:1].expand_as(group)), e


@pytest.mark.parametrize("rows", [1, 33, 128, 129, 176, 255, 256])
@pytest.mark.parametrize("layout,K,N", [("k_contiguous", 1024, 1280), ("n_contiguous", 1024, 1280), ("k_contiguous", 64, 8), ("k_contiguous", 1000, 264)])
def test_grouped_gemm_single_tile_groups(dev, oracle, rows, layout, K, N):
    """Groups of one row tile walk the K tiles from a start of their own: every start, one K tile in all, a partial last one."""
    ops = _ops()
    torch.manual_seed(22)
    E = 4
    counts = [rows, 0, 1, rows]
    sei = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    ssi = torch.randperm(sum(counts), generator=torch.Generator().manual_seed(3))
    X, W = torch.randn(sum(counts), K).bfloat16(), (torch.randn(E, K, N) * 0.05).bfloat16()
    Wd = W.permute(0, 2, 1).contiguous().to(dev).permute(0, 2, 1) if layout == "k_contiguous" else W.to(dev)
    y = ops.scatter2scatter(X.to(dev), Wd, sei.to(dev), ssi.to(dev), 1)
    ref = oracle.scatter2scatter_lora(X, W, None, None, 0, sei, ssi, 1)
    # one bf16 rounding of fp32 sums: half an ulp, 2^-9 of the value, and the sum's own error far below it
    assert float((y.float().cpu() - ref).abs().max()) <= 2.0 ** -8 * float(ref.abs().max())


@pytest.mark.parametrize("K,N", [(544, 2080), (1056, 96), (32, 544)])
@pytest.mark.parametrize("r", [16, 17, 32, 33, 80])
def test_group_bwd_ab_of_several_rank_chunks(dev, oracle, K, N, r):
    """Up to two chunks of 16 rank columns, with both products of each, share a launch: partial chunks, an odd number of them, and
    products of very different widths (one or several column blocks, K and N on either side)."""
    ops = _ops()
    torch.manual_seed(r)
    counts = torch.tensor([257, 0, 31, 1])
    eo, R, E = counts.cumsum(0), int(counts.sum()), len(counts)
    X, DY = torch.randn(R, K).bfloat16(), torch.randn(R, N).bfloat16()
    A, B = (torch.randn(E, K, r) * 0.1).bfloat16(), (torch.randn(E, r, N) * 0.1).bfloat16()
    dA, dB = ops.group_bwd_AB(DY.to(dev), X.to(dev), A.to(dev), B.to(dev), 2.0, eo.to(dev), E)
    dAo, dBo = oracle.group_bwd_AB(DY, X, A, B, 2.0, eo, E)
    check_expert_grads(dA, dAo, TOL[torch.bfloat16] * 1.5, "dA"); check_expert_grads(dB, dBo, TOL[torch.bfloat16] * 1.5, "dB")


@pytest.mark.parametrize("K,N,r", [(72, 64, 5), (1000, 264, 20), (200, 128, 100), (256, 320, 96)])
def test_scatter2scatter_lora_packs_any_width_and_rank(dev, oracle, K, N, r):
    """The pack launch takes up to six chunks of both factors: widths that are no whole fragment, ranks that need two launches."""
    ops = _ops()
    torch.manual_seed(r)
    sei = torch.tensor([0] * 130 + [1] * 3 + [3] * 40)
    ssi = torch.randperm(len(sei))
    X, W = torch.randn(len(sei), K).bfloat16(), (torch.randn(4, K, N) * 0.05).bfloat16()
    A, B = (torch.randn(4, K, r) * 0.1).bfloat16(), (torch.randn(4, r, N) * 0.1).bfloat16()
    for Ad, Bd in ((A.to(dev), B.to(dev)), (A.permute(0, 2, 1).contiguous().to(dev).permute(0, 2, 1), B.permute(0, 2, 1).contiguous().to(dev).permute(0, 2, 1))):
        y = ops.scatter2scatter_lora(X.to(dev), W.to(dev), Ad, Bd, 0.5, sei.to(dev), ssi.to(dev), 1, None)
        ref = oracle.scatter2scatter_lora(X, W, A, B, 0.5, sei, ssi, 1)
        assert rel(y, ref) < TOL[torch.bfloat16]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("K", [1, 15, 63, 64, 65, 127, 128, 129, 130, 257])
@pytest.mark.parametrize("layout", ["k_contiguous", "n_contiguous"])
def test_generic_kernels_at_the_edges_of_a_contraction_step(dev, oracle, dtype, K, layout):
    """The kernels of the sizes that the matrix cores do not take, at contractions of one step, one step more or less and a few: the
    product with adapters, and the per-expert product over rows (whose contraction is the group: 0, 1, 63 .. 130 rows)."""
    ops = _ops()
    torch.manual_seed(K)
    counts, N, r = [63, 0, 64, 1, 65, 130], 19, 3
    E, R = len(counts), sum(counts)
    sei = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    ssi = torch.randperm(R)
    X, W = torch.randn(R, K).to(dtype), (torch.randn(E, K, N) * 0.3).to(dtype)
    A, B = (torch.randn(E, K, r) * 0.3).to(dtype), (torch.randn(E, r, N) * 0.3).to(dtype)
    Wd = W.permute(0, 2, 1).contiguous().to(dev).permute(0, 2, 1) if layout == "k_contiguous" else W.to(dev)
    y = ops.scatter2scatter_lora(X.to(dev), Wd, A.to(dev), B.to(dev), 2.0, sei.to(dev), ssi.to(dev), 1, None)
    ref = oracle.scatter2scatter_lora(X, W, A, B, 2.0, sei, ssi, 1)
    assert rel(y, ref) < TOL[dtype]
    dy = torch.randn(R, N).to(dtype)
    dw = ops.group_bwd_W(dy.to(dev), X.to(dev), torch.tensor(counts).cumsum(0).to(dev), E)
    at = torch.tensor([0] + counts).cumsum(0)
    want = torch.stack([X[a:b].float().t() @ dy[a:b].float() for a, b in zip(at[:-1], at[1:])])
    check_expert_grads(dw, want, TOL[dtype])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,E,k,K,N,r,gates,layout", [
    (333, 4, 2, 256, 384, 16, True, "k_contiguous"), (100, 3, 1, 64, 96, 8, False, "k_contiguous"), (257, 5, 3, 96, 160, 24, True, "n_contiguous"),
    (64, 2, 2, 128, 64, 33, False, "n_contiguous"), (700, 6, 4, 320, 64, 64, True, "k_contiguous"), (257, 5, 3, 96, 160, 24, False, "n_contiguous"),
    (700, 6, 4, 320, 64, 64, False, "k_contiguous"), (90, 3, 2, 64, 64, 65, True, "k_contiguous"),
    (40, 3, 2, 48, 64, 16, True, "k_contiguous"), (50, 2, 2, 64, 32, 16, False, "k_contiguous")])
def test_projection_backward_on_gathered_rows(dev, oracle, dtype, T, E, k, K, N, r, gates, layout):
    """The backward pass that reads dY and X where they lie, on both sides of its rule (ranks to 64, contractions of at least 64 and multiples of
    32, gates with bf16 rows only; the last three, and in fp16 the gated ones, take the route over gathered copies): adapter gradients, dX and the gates' against the fp32 oracle."""
    import moe_distributed_training_amd as moe
    torch.manual_seed(T + r)
    _, sei, ssi, eo = _routing(oracle, T, E, k, T, skew=True)
    X = torch.randn(T, K).to(dtype)
    W = (torch.randn(E, N, K) * 0.05).to(dtype).permute(0, 2, 1) if layout == "k_contiguous" else (torch.randn(E, K, N) * 0.05).to(dtype)
    A, B = (torch.randn(E, K, r) * 0.05).to(dtype), (torch.randn(E, r, N) * 0.05).to(dtype)
    G = torch.rand(T, k).to(dtype) if gates else None
    dY = torch.randn(T if gates else T * k, N).to(dtype)
    f32 = lambda t: None if t is None else t.float().clone().requires_grad_(True)
    Xo, Ao, Bo, Go = f32(X), f32(A), f32(B), f32(G)
    oracle.parallel_linear_lora(Xo, W.float(), Ao, Bo, r, 32.0, k, sei, ssi, None, eo, Go, False, False).backward(dY.float())
    d = lambda t: None if t is None else t.detach().to(dev).requires_grad_(True)
    Xd, Ad, Bd, Gd = d(X), d(A), d(B), d(G)
    Wd = W.permute(0, 2, 1).contiguous().to(dev).permute(0, 2, 1) if layout == "k_contiguous" else W.to(dev)
    pb, eod = moe.padded_block_indices(sei.to(dev), E)
    moe.parallel_linear_lora(Xd, Wd, Ad, Bd, r, 32.0, k, sei.to(dev), ssi.to(dev), pb, eod, Gd, False, False).backward(dY.to(dev))
    tol = TOL[dtype] * 1.5
    assert rel(Xd.grad, Xo.grad) < tol
    check_expert_grads(Ad.grad, Ao.grad, tol, "dA"); check_expert_grads(Bd.grad, Bo.grad, tol, "dB")
    if gates:
        assert rel(Gd.grad, Go.grad) < tol


@pytest.mark.parametrize("hooked", [False, True])
def test_projection_backward_of_gated_fp16_rows_near_the_largest_number(dev, oracle, hooked):
    """dY of up to 3e4 under gates of 1e-3: dY B^T alone passes 65504, every gradient is finite, as the product of the weighted rows is; and the same
    where a saved-tensor hook hands the gates back with other strides."""
    import moe_distributed_training_amd as moe
    torch.manual_seed(3)
    T, E, k, K, N, r = 64, 2, 2, 256, 256, 16
    _, sei, ssi, eo = _routing(oracle, T, E, k, T)
    h = lambda *s: torch.randn(*s)
    X, W, A, B = h(T, K).half(), (h(E, K, N) * 0.02).half(), (h(E, K, r) * 0.1).half(), h(E, r, N).half()
    G, dY = 1e-3 * (0.5 + torch.rand(T, k)), ((torch.rand(T, N) * 2 - 1) * 3e4).half()
    f32 = lambda t: t.float().clone().requires_grad_(True)
    Xo, Ao, Bo, Go = f32(X), f32(A), f32(B), f32(G)
    oracle.parallel_linear_lora(Xo, W.float(), Ao, Bo, r, 32.0, k, sei, ssi, None, eo, Go, False, False).backward(dY.float())
    Xd, Ad, Bd, Gd = (t.to(dev).requires_grad_(True) for t in (X, A, B, G))
    pb, eod = moe.padded_block_indices(sei.to(dev), E)
    turn = lambda t: t.t().contiguous().t() if hooked and t.shape == (T, k) else t   # (the gates; same values, strides (1, T))
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, turn):
        y = moe.parallel_linear_lora(Xd, W.to(dev), Ad, Bd, r, 32.0, k, sei.to(dev), ssi.to(dev), pb, eod, Gd, False, False)
        y.backward(dY.to(dev))
    tol = TOL[torch.float16] * 1.5
    for got, want in ((Xd, Xo), (Ad, Ao), (Bd, Bo), (Gd, Go)):
        assert torch.isfinite(got.grad).all() and rel(got.grad, want.grad) < tol


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("k,n_extra,cols", [(1, 1, 64), (2, 8, 4096), (3, 9, 72), (4, 64, 1032), (8, 33, 2048), (0, 16, 256), (2, 1025, 64)])
def test_combine_with_a_dense_tail(dev, dtype, k, n_extra, cols):
    """The fan-out sum with the router's input gradient behind it, by the matrix instructions' kernel (16 tokens and 128 columns per wave; three
    tokens more than a whole number of groups, columns and tail rows that fill neither) and by one token per workgroup: against 64 bits, and a
    token's sum does not depend on the tokens around it."""
    from moe_distributed_training_amd._lib import lib, check, ptr, stream_ptr, dtype_code
    T = 4 * torch.cuda.get_device_properties(dev).multi_processor_count + 3
    g = torch.Generator(device=dev).manual_seed(k + n_extra)
    y = torch.randn(max(1, T * k), cols, generator=g, device=dev).to(dtype)
    rows, coef = torch.randn(n_extra, cols, generator=g, device=dev).to(dtype), torch.randn(T, n_extra, generator=g, device=dev)

    def run(t0, t1):
        out = torch.empty(t1 - t0, cols, dtype=dtype, device=dev)
        c = coef[t0:t1].contiguous()
        check(lib.moe_combine(ptr(y[t0 * k:]) if k else None, cols, ptr(out), cols, None, 0, None, k, t1 - t0, cols, dtype_code(y), ptr(c), ptr(rows), cols,
                              n_extra, stream_ptr(dev)), "moe_combine")
        return out
    whole = run(0, T)
    step = 200
    pieces = torch.cat([run(t, min(T, t + step)) for t in range(0, T, step)])
    assert torch.equal(whole, pieces)
    want = coef.double() @ rows.double() + (y.double().view(T, k, cols).sum(1) if k else 0.0)
    assert rel(whole, want) < TOL[dtype]




@pytest.mark.parametrize("T,E,k,K,N", [(1, 1, 1, 1, 1), (40, 3, 2, 63, 17), (33, 5, 3, 64, 16), (100, 4, 2, 130, 250), (7, 40, 8, 65, 33)])
def test_gate_and_up_in_one_launch_fp32(dev, oracle, T, E, k, K, N):
    """moe_swiglu_pair against the three launches it stands for, bit for bit, at contractions and columns on both sides of its tiles and with
    experts without rows; and that other types, which round in between, are refused."""
    from moe_distributed_training_amd._lib import lib, check, ptr, stream_ptr
    ops = _ops()
    torch.manual_seed(T + K)
    _, sei, ssi, eo = _routing(oracle, T, E, k, skew=True)
    x, w1, w3 = torch.randn(T, K, device=dev), torch.randn(E, N, K, device=dev) * 0.1, torch.randn(E, N, K, device=dev) * 0.1
    p, o, s = ssi.to(dev), eo.to(dev), sei.to(dev)
    gate, up = (ops.scatter2scatter(x, w.permute(0, 2, 1), s, p, k, None, False, True) for w in (w1, w3))
    want, h = torch.empty_like(gate), torch.full_like(gate, -7.0)
    check(lib.moe_swiglu(ptr(gate), ptr(up), ptr(want), gate.numel(), 2, stream_ptr(dev)), "moe_swiglu")
    args = lambda dt: (ptr(x), K, 1, ptr(w1), ptr(w3), N * K, 1, K, ptr(h), N, ptr(p), int(p.dtype == torch.int64), ptr(o), int(o.dtype == torch.int64), E, T * k, K, N,
                       k, dt, stream_ptr(dev))
    assert lib.moe_swiglu_pair(*args(0)) == -2
    check(lib.moe_swiglu_pair(*args(2)), "moe_swiglu_pair")
    assert torch.equal(h, want)


def _us(fn, n=20):
    """GPU time of a call in us, best of five replays of n calls in a graph (no host work between the calls)."""
    fn()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for _ in range(n):
            fn()
    times = []
    for _ in range(6):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        graph.replay()
        b.record()
        torch.cuda.synchronize()
        times.append(a.elapsed_time(b) / n * 1e3)
    return min(times[1:])


def test_products_over_few_rows_are_not_worked_through_as_over_many(dev):
    """One row per expert against 64 (2048 x 2048, fp32: 90 and 264 us; 261 and 264 when a step of 64 rows was always worked through)."""
    ops = _ops()
    E, N = 8, 2048

    def product(rows):
        dy, x = torch.randn(E * rows, N, device=dev), torch.randn(E * rows, N, device=dev)
        off = torch.arange(1, E + 1, device=dev) * rows
        return _us(lambda: ops.group_bwd_W(dy, x, off, E))
    one, many = product(1), product(64)
    assert one < 0.6 * many, (one, many)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("K", [7, 16, 17, 31, 32, 33])
def test_short_contractions_of_the_generic_product(dev, oracle, dtype, K):
    """Contractions on both sides of the line between steps of 16 and of 64, with and without adapters, weights and factors of either
    orientation (which choose the direction of the loads)."""
    ops = _ops()
    torch.manual_seed(K)
    counts, N, r = [17, 0, 1, 40], 21, 5
    E, R = len(counts), sum(counts)
    sei, ssi = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)), torch.randperm(R)
    X, W = torch.randn(R, K).to(dtype), torch.randn(E, K, N).to(dtype)
    A, B = (torch.randn(E, K, r) * 0.3).to(dtype), (torch.randn(E, r, N) * 0.3).to(dtype)
    turned = lambda t: t.transpose(1, 2).contiguous().to(dev).transpose(1, 2)
    for w in (W.to(dev), turned(W)):
        assert rel(ops.scatter2scatter(X.to(dev), w, sei.to(dev), ssi.to(dev), 1), oracle.scatter2scatter_lora(X, W, torch.zeros_like(A), B, 1.0, sei, ssi, 1)) < TOL[dtype]
        for a in (A.to(dev), turned(A)):
            for b in (B.to(dev), turned(B)):
                y = ops.scatter2scatter_lora(X.to(dev), w, a, b, 2.0, sei.to(dev), ssi.to(dev), 1, None)
                assert rel(y, oracle.scatter2scatter_lora(X, W, A, B, 2.0, sei, ssi, 1)) < TOL[dtype]


def test_a_projection_of_few_columns_is_not_worked_through_as_of_many(dev):
    """2048 rows, 8 columns against 64 (to 2048, fp32: 27 and 45 us; 46 and 45 when a step of 64 columns was always worked through)."""
    ops = _ops()
    E, R = 8, 2048
    sei, ssi = torch.arange(E, device=dev).repeat_interleave(R // E), torch.arange(R, device=dev)

    def projection(K):
        x, w = torch.randn(R, K, device=dev), torch.randn(E, 2048, K, device=dev).permute(0, 2, 1)
        return _us(lambda: ops.scatter2scatter(x, w, sei, ssi, 1))
    few, many = projection(8), projection(64)
    assert few < 0.8 * many, (few, many)


def test_factors_decide_the_direction_of_the_generic_product(dev):
    """Adapters contiguous along the output beside weights contiguous along the contraction: 145 us with loads along the output, 584 with
    loads along the contraction, 122 with both contiguous along the output."""
    ops = _ops()
    E, K, N, r, T = 8, 256, 512, 16, 2048
    x, w = torch.randn(T, K, device=dev), torch.randn(E, N, K, device=dev).permute(0, 2, 1)
    a, b = torch.randn(E, K, r, device=dev), torch.randn(E, r, N, device=dev)
    sei, ssi = torch.arange(E, device=dev).repeat_interleave(T // E), torch.randperm(T, device=dev)
    time = lambda w: _us(lambda: ops.scatter2scatter_lora(x, w, a, b, 1.0, sei, ssi, 1, None))
    along_k, along_n = time(w), time(w.contiguous())
    assert along_k < 1.8 * along_n, (along_k, along_n)


def test_few_rows_of_tail_cost_a_large_sum_little(dev):
    """8192 tokens of 8 rows, d=4096: 105 us without a tail, 120 with one of eight rows, 160 where the rows are fetched by the tail's kernel."""
    ops = _ops()
    T, k, d = 8192, 8, 4096
    y = torch.randn(T * k, d, device=dev).bfloat16()
    rows, coef = torch.randn(8, d, device=dev).bfloat16(), torch.randn(T, 8, device=dev)
    plain, tailed = _us(lambda: ops.combine(y, None, None, k)), _us(lambda: ops.combine(y, None, None, k, None, coef, rows))
    assert tailed < 1.3 * plain, (tailed, plain)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("gates", [None, torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,k,n_extra,cols", [(19, 1, 24, 2056), (35, 3, 33, 4104), (18, 8, 64, 1024), (50, 2, 8, 72), (33, 8, 130, 4096)])
def test_weighted_sum_of_gathered_rows_with_a_tail(dev, dtype, gates, T, k, n_extra, cols):
    """The fan-out sum of rows that a permutation names, with weights of any type and a dense tail, by the tail's kernel (long tails) and one token
    per workgroup: tokens past a whole group of 16, columns past 128 and 512, against 64 bits."""
    ops = _ops()
    g = torch.Generator(device=dev).manual_seed(T)
    y, inv = torch.randn(T * k, cols, generator=g, device=dev).to(dtype), torch.randperm(T * k, generator=g, device=dev).int()
    w = None if gates is None else torch.rand(T, k, generator=g, device=dev).to(gates)
    rows, coef = torch.randn(n_extra, cols, generator=g, device=dev).to(dtype), torch.randn(T, n_extra, generator=g, device=dev)
    got = ops.combine(y, w, inv, k, None, coef, rows)
    picked = y.double()[inv.long()].view(T, k, cols)
    want = (picked if w is None else picked * w.double()[:, :, None]).sum(1) + coef.double() @ rows.double()
    assert rel(got, want) < TOL[dtype]


@pytest.mark.parametrize("dtype,K,N,r", [(torch.float32, 64, 96, 8), (torch.float16, 64, 96, 8), (torch.bfloat16, 64, 96, 72), (torch.bfloat16, 48, 96, 8), (torch.bfloat16, 64, 32, 8)])
def test_projection_backward_allocates_nothing_for_the_route_that_refuses(dev, oracle, dtype, K, N, r):
    """Gated projections that the backward on gathered rows does not take by their type or sizes: dY and X grouped, the adapters' gradients, two workspaces, the
    gates' gradient and the fan-out sum, and no buffers of the other route."""
    import moe_distributed_training_amd as moe
    T, E, k = 40, 3, 2
    _, sei, ssi, eo = _routing(oracle, T, E, k)
    g = lambda *s: (torch.randn(*s, device=dev) * 0.1).to(dtype).requires_grad_(True)
    x, W, A, B, G = g(T, K), g(E, K, N).detach(), g(E, K, r), g(E, r, N), g(T, k)
    y = moe.parallel_linear_lora(x, W, A, B, r, 32.0, k, sei.to(dev), ssi.to(dev), None, eo.to(dev), gates=G)
    dy = torch.randn_like(y)
    count = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]
    n = count()
    grads = torch.autograd.grad(y, (x, A, B, G), dy)
    assert count() - n == 8 and len(grads) == 4
