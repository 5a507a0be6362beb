"""The many-token kernel (fp32 X of more than 16 tokens): against the oracle at the edges of its tiles — tokens around
its groups of 16 and 64, rows around its 256 columns, one superblock, K cut over workgroups and not — and its prologue,
epilogue and residual against the same call as separate launches."""
import numpy as np
import pytest

from test_gpu_fused import gpu  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu

Q4_K, Q5_K, Q6_K = 12, 13, 14


@pytest.mark.parametrize("type_", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("M,N,K", [(17, 1, 256), (32, 255, 512), (33, 257, 2816), (64, 300, 1024), (65, 256, 256),
                                   (129, 520, 4096), (9, 61500, 256), (16, 65537, 256)])
def test_many_tokens_vs_oracle(gpu, kqo, type_, M, N, K):  # noqa: F811
    from backpack_amd import capi, kquant
    print("wide", type_, M, N, K, flush=True)
    raw, packed, w = gpu.make_weight(type_, N, K, seed=M + N)
    rng = np.random.default_rng(K + M)
    X = rng.standard_normal((M, K)).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32)
    capi.force_kernel(8)
    try:
        got = kquant.matmul(gpu.dev(X), w, bias=gpu.dev(bias)).cpu().numpy()
    finally:
        capi.force_kernel(0)
    assert (capi.last_kernel(), capi.last_form()) == ("mtile", "many_token")
    # hi + lo keep 22 bits of x: 2^-22 of the largest element per product, far inside the slack of the tile kernels
    gpu.check_matmul(kqo, type_, got, X, packed, N, K, bias=bias, label="wide", slack=1e-5)
    # rows do not depend on their neighbours: one token's row is the same from a group of another size (fewer tokens:
    # another number of splits may add K in another order, one fp32 rounding per split)
    capi.force_kernel(8)
    try:
        one = kquant.matmul(gpu.dev(X[:1]), w, bias=gpu.dev(bias)).cpu().numpy()
    finally:
        capi.force_kernel(0)
    rms = float(np.sqrt(np.mean(got.astype(np.float64) ** 2)))
    assert float(np.abs(one[0] - got[0]).max()) <= 2e-6 * rms + 2e-6 * float(np.abs(got[0]).max())


@pytest.mark.parametrize("type_", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("M", [17, 48, 64])
@pytest.mark.parametrize("blocks", [1, 2, 3, 4, 5, 7])
def test_walks_of_few_superblocks(gpu, kqo, type_, M, blocks):  # noqa: F811
    """Every place in the ring of half superblocks as the last one, one workgroup's rows and a ragged second."""
    from backpack_amd import capi, kquant
    N, K = 270, 256 * blocks
    raw, packed, w = gpu.make_weight(type_, N, K, seed=blocks)
    X = np.random.default_rng(M).standard_normal((M, K)).astype(np.float32)
    capi.force_kernel(8)
    capi.set_option("gemv_splits", 1)
    try:
        got = kquant.matmul(gpu.dev(X), w).cpu().numpy()
    finally:
        capi.force_kernel(0)
        capi.set_option("gemv_splits", 0)
    gpu.check_matmul(kqo, type_, got, X, packed, N, K, label="walk", slack=1e-5)


@pytest.mark.parametrize("type_", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("M,blocks", [(17, 1), (48, 2), (64, 3)])
def test_several_row_groups_per_workgroup(gpu, kqo, type_, M, blocks):  # noqa: F811
    """More groups of 256 rows than CUs: a workgroup walks two, the last of them ragged.  Windows of rows at both
    ends and in the middle, with a bias and, in place, a residual."""
    from backpack_amd import capi, kquant, synth
    N, K = 256 * 299 + 7, 256 * blocks
    print("groups", type_, M, N, K, flush=True)
    raw, packed, w = gpu.make_weight(type_, N, K, seed=blocks)
    rng = np.random.default_rng(M)
    X = rng.standard_normal((M, K)).astype(np.float32)
    bias, res = rng.standard_normal(N).astype(np.float32), rng.standard_normal((M, N)).astype(np.float32)
    got = kquant.matmul(gpu.dev(X), w, bias=gpu.dev(bias)).cpu().numpy()
    assert capi.last_form() == "many_token"
    y = gpu.dev(res)
    kquant.matmul_fused(gpu.dev(X), w, residual=y, out=y)
    y = y.cpu().numpy()
    words = synth.row_stride_words(type_, K)
    for a, b in ((0, 300), (256 * 149 - 20, 256 * 150 + 20), (N - 530, N)):
        rows = packed[a * words:b * words]
        gpu.check_matmul(kqo, type_, np.ascontiguousarray(got[:, a:b]), X, rows, b - a, K, bias=bias[a:b], label="groups", slack=1e-5)
        # the residual is added to the same product, one rounding each
        plain = got[:, a:b].astype(np.float64) - bias[a:b]
        tol = 4e-7 * (np.abs(got[:, a:b]) + np.abs(bias[a:b]) + np.abs(res[:, a:b]) + np.abs(plain))
        assert np.all(np.abs(y[:, a:b] - (plain + res[:, a:b])) <= tol)


@pytest.mark.parametrize("tgu,tdn", [(Q4_K, Q6_K), (Q5_K, Q4_K), (Q6_K, Q5_K)])
@pytest.mark.parametrize("T,H,I", [(80, 256, 1792), (80, 3328, 256), (320, 512, 2304), (320, 3328, 512)])
def test_moe_several_row_groups_per_workgroup(gpu, kqo, tgu, tdn, T, H, I):  # noqa: F811
    """64 experts of 5 or 20 pairs and 13 to 18 groups of rows: a workgroup walks several of a record's, the last one
    fewer.  A few tokens against the oracle, all against the 16-token tile kernel."""
    from backpack_amd import capi, kquant
    print("moe groups", tgu, tdn, T, H, I, flush=True)
    E, k = 64, 4
    _, gp, gw = gpu.make_weight(tgu, E * I, H, seed=31)
    _, up, uw = gpu.make_weight(tgu, E * I, H, seed=32)
    _, dp, dw = gpu.make_weight(tdn, E * H, I, seed=33)
    rng = np.random.default_rng(T + H)
    eidx = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.uint32)
    ew = rng.random((T, k)).astype(np.float32)
    X = (rng.standard_normal((T, H)) * 0.1).astype(np.float32)
    args = (gpu.dev(X), gw, uw, dw, gpu.dev(eidx.view(np.int32)), gpu.dev(ew), E)
    capi.force_kernel(8)
    try:
        got = kquant.moe_ffn(*args).cpu().numpy()
        capi.force_kernel(6)
        tile = kquant.moe_ffn(*args).cpu().numpy()
    finally:
        capi.force_kernel(0)
    sel = rng.choice(T, 4, replace=False)
    want = kqo.moe_ffn(tgu, tdn, X[sel], gp, up, dp, eidx[sel], ew[sel], H, I)
    rms = float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))
    assert np.all(np.abs(got[sel] - want) <= 1e-3 * rms + 1e-3 * np.abs(want))
    assert np.abs(got - tile).max() <= 1e-4 * rms + 1e-4 * np.abs(tile).max()


@pytest.mark.parametrize("type_,M,N,K,pro,epi,res", [(Q4_K, 48, 272, 512, 1, 2, False), (Q5_K, 17, 136, 4096, 1, 3, False),
                                                     (Q6_K, 70, 257, 1024, 2, 0, True), (Q4_K, 21, 96, 256, 3, 0, True)])
def test_many_tokens_fused_vs_separate(gpu, type_, M, N, K, pro, epi, res):  # noqa: F811
    from backpack_amd import capi, kquant
    print("wide fused", type_, M, N, K, pro, epi, res, flush=True)
    raw, packed, w = gpu.make_weight(type_, 2 * N if epi else N, K, seed=M)
    rng = np.random.default_rng(M)
    x = gpu.dev(rng.standard_normal((M, 2 * K if pro >= 2 else K)).astype(np.float32))
    nw = gpu.dev(rng.standard_normal(K).astype(np.float32)) if pro == 1 else None
    r = gpu.dev(rng.standard_normal((M, N)).astype(np.float32)) if res else None
    a = kquant.matmul_fused(x, w, pro, norm_w=nw, eps=1e-5, residual=r, epilogue=epi).cpu().numpy()
    assert capi.last_form() == "many_token"
    if res:   # in place: the residual is the output buffer
        y = r.clone()
        kquant.matmul_fused(x, w, pro, norm_w=nw, eps=1e-5, residual=y, out=y)
        assert np.array_equal(y.cpu().numpy(), a)
    capi.set_option("fused_separate", 1)
    try:
        b = kquant.matmul_fused(x, w, pro, norm_w=nw, eps=1e-5, residual=r, epilogue=epi).cpu().numpy()
    finally:
        capi.set_option("fused_separate", 0)
    rms = float(np.sqrt(np.mean(b.astype(np.float64) ** 2)))
    assert np.isfinite(a).all()
    # the same split products from x that differs by the rounding of its norm (a few 2^-24)
    assert float(np.abs(a - b).max()) <= 1e-5 * rms + 1e-5 * float(np.abs(b).max())


@pytest.mark.parametrize("K,M,form", [(253440, 65, "tile"), (256000, 63, "wide")])
def test_rows_too_long_for_steps_of_64_tokens(gpu, kqo, K, M, form):  # noqa: F811
    """Rows so long that fewer than 64 tokens of split X fit the scratch: more tokens than fit go to the tile kernel
    (the forced family says that it cannot), a call that fits whole stays."""
    from backpack_amd import capi, kquant
    print("long rows", K, M, flush=True)
    raw, packed, w = gpu.make_weight(Q4_K, 3, K, seed=M)
    X = np.random.default_rng(M).standard_normal((M, K)).astype(np.float32)
    got = kquant.matmul(gpu.dev(X), w).cpu().numpy()
    gpu.check_matmul(kqo, Q4_K, got, X, packed, 3, K, label="long rows", slack=1e-5)
    capi.force_kernel(8)
    try:
        if form == "wide":
            kquant.matmul(gpu.dev(X), w)
        else:
            with pytest.raises(capi.BpkError) as e:
                kquant.matmul(gpu.dev(X), w)
            assert e.value.code == -2
    finally:
        capi.force_kernel(0)


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("type_,M,N,K,pro,epi", [(Q4_K, 33, 272, 1024, 1, 2), (Q5_K, 17, 129, 768, 0, 3), (Q6_K, 50, 200, 1024, 1, 3), (Q6_K, 64, 16, 2816, 0, 2)])
def test_many_tokens_epilogue_with_bias_vs_oracle(gpu, kqo, type_, M, N, K, pro, epi, splits):  # noqa: F811
    """act(gate) * up with a bias under it, outputs that are no multiple of a wave's 16, K in one piece (the kernel's own
    store) and cut (the launch that adds the splits)."""
    from backpack_amd import capi, kquant
    print("wide epilogue", type_, M, N, K, pro, epi, splits, flush=True)
    raw, packed, w = gpu.make_weight(type_, 2 * N, K, seed=N)
    rng = np.random.default_rng(N + splits)
    x = rng.standard_normal((M, K)).astype(np.float32)
    nw = (1 + 0.1 * rng.standard_normal(K)).astype(np.float32) if pro else None
    bias = rng.standard_normal(2 * N).astype(np.float32)
    capi.force_kernel(8)
    capi.set_option("gemv_splits", splits)
    try:
        got = kquant.matmul_fused(gpu.dev(x), w, pro, norm_w=gpu.dev(nw) if pro else None, eps=1e-5, bias=gpu.dev(bias), epilogue=epi).cpu().numpy()
    finally:
        capi.force_kernel(0)
        capi.set_option("gemv_splits", 0)
    assert capi.last_form() == "many_token"
    xp = kqo.prologue(pro, x, K, norm_w=nw, eps=1e-5) if pro else x
    want = kqo.prologue(epi, kqo.matmul(type_, xp, packed, 2 * N, K, bias=bias), N)
    # the product of two matvec results, each good to ~1e-6 of its rms, as in the decode forms' test
    rms = float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))
    assert np.all(np.abs(got - want) <= 2e-4 * (rms + np.abs(want))), float(np.abs(got - want).max())


@pytest.mark.parametrize("type_,pro,res", [(Q4_K, 0, False), (Q6_K, 1, True), (Q5_K, 2, True)])
def test_more_tokens_than_the_scratch_holds(gpu, kqo, type_, pro, res):  # noqa: F811
    """1140 tokens of 14336 elements: the split X goes through the 64 MiB of scratch in two steps, of 1088 and of 52 tokens;
    the rows around the border and at both ends against the oracle, a residual that is the output buffer."""
    from backpack_amd import capi, kquant
    M, N, K = 1140, 19, 14336
    assert (64 << 20) // (1060 * (K // 256)) // 64 * 64 == 1088
    print("wide steps", type_, pro, res, flush=True)
    raw, packed, w = gpu.make_weight(type_, N, K, seed=5)
    rng = np.random.default_rng(pro)
    x = rng.standard_normal((M, 2 * K if pro == 2 else K), dtype=np.float32)
    nw = (1 + 0.1 * rng.standard_normal(K)).astype(np.float32) if pro == 1 else None
    bias = rng.standard_normal(N).astype(np.float32)
    r = rng.standard_normal((M, N)).astype(np.float32) if res else None
    if pro or res:
        y = gpu.dev(r)
        kquant.matmul_fused(gpu.dev(x), w, pro, norm_w=gpu.dev(nw) if pro == 1 else None, eps=1e-5, residual=y, bias=gpu.dev(bias), out=y)
    else:
        y = kquant.matmul(gpu.dev(x), w, bias=gpu.dev(bias))
    assert capi.last_form() == "many_token"
    sel = np.r_[0:4, 1084:1092, 1136:1140]
    xs = x[sel] if pro == 0 else kqo.prologue(pro, x[sel], K, norm_w=nw, eps=1e-5)
    got = y.cpu().numpy()[sel] - (r[sel] if res else 0.0)
    # (the residual's subtraction here rounds once more: 2^-24 of outputs of up to some 10 of their rms)
    gpu.check_matmul(kqo, type_, got, xs, packed, N, K, bias=bias, label="steps", slack=1e-5)


@pytest.mark.parametrize("type_", [Q4_K, Q5_K, Q6_K])
def test_an_outlier_costs_no_more_than_on_the_tile_kernel(gpu, kqo, type_):  # noqa: F811
    """A superblock accumulates in one chain of matrix instructions: beside an activation 10^4 times the others the error
    against 64 bits stays below the 16-token tile kernel's, which adds up after every 32 elements (measured: a third to a
    twentieth of it)."""
    from backpack_amd import capi, kquant
    M, N, K = 20, 300, 1024
    raw, packed, w = gpu.make_weight(type_, N, K, seed=6)
    X = np.random.default_rng(6).standard_normal((M, K)).astype(np.float32)
    X[:, 5], X[:, 700] = 1e4, -1e4
    want = kqo.matmul_f64(type_, X, packed, N, K)
    err = {}
    try:
        for family in (6, 8):
            capi.force_kernel(family)
            err[family] = float(np.linalg.norm(kquant.matmul(gpu.dev(X), w).cpu().numpy() - want) / np.linalg.norm(want))
    finally:
        capi.force_kernel(0)
    assert err[8] < err[6] and err[8] < 4e-6, err


# few pairs per expert (records of 16: every launch is one round of the CUs), a skewed routing, one slot per token (whose
# split X does not fit beside the records: the 16-token tile kernel)
@pytest.mark.parametrize("tgu,tdn,T,E,k,H,I,skew", [(Q4_K, Q6_K, 5, 8, 2, 256, 256, False), (Q4_K, Q6_K, 17, 2, 2, 512, 256, False),
                                                    (Q5_K, Q5_K, 65, 4, 2, 768, 512, False), (Q6_K, Q4_K, 200, 8, 3, 512, 768, True),
                                                    (Q4_K, Q4_K, 300, 4, 2, 256, 512, False), (Q4_K, Q6_K, 40, 4, 1, 512, 256, False),
                                                    (Q5_K, Q6_K, 40, 4, 1, 1280, 256, False)])
def test_moe_ffn_many_pairs_vs_oracle(gpu, kqo, tgu, tdn, T, E, k, H, I, skew):  # noqa: F811
    from backpack_amd import capi, kquant
    print("wide moe", tgu, tdn, T, E, k, H, I, skew, flush=True)
    _, gp, gw = gpu.make_weight(tgu, E * I, H, seed=81)
    _, up, uw = gpu.make_weight(tgu, E * I, H, seed=82)
    _, dp, dw = gpu.make_weight(tdn, E * H, I, seed=83)
    rng = np.random.default_rng(T)
    eidx = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.uint32)
    if skew:   # every token's first slot is expert 3: one expert of many records beside experts of few
        eidx[:, 1:][eidx[:, 1:] == 3] = 0
        eidx[:, 0] = 3
    ew = rng.random((T, k)).astype(np.float32)
    X = (rng.standard_normal((T, H)) * 0.1).astype(np.float32)
    args = (gpu.dev(X), gw, uw, dw, gpu.dev(eidx.view(np.int32)), gpu.dev(ew), E)
    got = kquant.moe_ffn(*args).cpu().numpy()
    assert (capi.last_kernel(), capi.last_form()) == ("moe_ffn_mtile", "" if k == 1 else "records_16")
    assert np.array_equal(got, kquant.moe_ffn(*args).cpu().numpy()), "a pair's result does not depend on its place"
    capi.force_kernel(6)
    try:
        tile = kquant.moe_ffn(*args).cpu().numpy()
    finally:
        capi.force_kernel(0)
    want = kqo.moe_ffn(tgu, tdn, X, gp, up, dp, eidx, ew, H, I)
    rms = float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))
    assert np.all(np.abs(got - want) <= 1e-3 * rms + 1e-3 * np.abs(want))
    # both split x into 22 bits of its superblock's largest: the sums' order is what differs
    assert np.abs(got - tile).max() <= 1e-4 * rms + 1e-4 * np.abs(want).max()


# enough pairs that records of 32, 48 and 64 save rounds; every type in both places, inter of two to four superblocks
@pytest.mark.parametrize("T,H,I,cap", [(600, 256, 512, 32), (600, 256, 1024, 48), (1300, 256, 512, 48), (1300, 512, 768, 64)])
@pytest.mark.parametrize("tgu,tdn", [(Q4_K, Q6_K), (Q5_K, Q5_K), (Q6_K, Q4_K)])
def test_moe_ffn_records_of_32_to_64_pairs(gpu, kqo, tgu, tdn, T, H, I, cap):  # noqa: F811
    """One expert whose pairs fill their records exactly, one with a pair more, one with three pairs, the rest on the
    last: some tokens against the oracle, all of them against the 16-token tile kernel."""
    from backpack_amd import capi, kquant
    print("records", tgu, tdn, T, H, I, cap, flush=True)
    E, k = 4, 2
    _, gp, gw = gpu.make_weight(tgu, E * I, H, seed=94)
    _, up, uw = gpu.make_weight(tgu, E * I, H, seed=95)
    _, dp, dw = gpu.make_weight(tdn, E * H, I, seed=96)
    rng = np.random.default_rng(T + cap)
    counts = [4 * cap, 4 * cap + 1, 3, T * k - 8 * cap - 4]
    eidx = rng.permutation(np.repeat(np.arange(E), counts)).astype(np.uint32).reshape(T, k)
    ew = rng.random((T, k)).astype(np.float32)
    X = (rng.standard_normal((T, H)) * 0.1).astype(np.float32)
    args = (gpu.dev(X), gw, uw, dw, gpu.dev(eidx.view(np.int32)), gpu.dev(ew), E)
    got = kquant.moe_ffn(*args).cpu().numpy()
    assert capi.last_form() == f"records_{cap}"
    assert np.array_equal(got, kquant.moe_ffn(*args).cpu().numpy()), "a pair's result does not depend on its place"
    capi.force_kernel(6)
    try:
        tile = kquant.moe_ffn(*args).cpu().numpy()
    finally:
        capi.force_kernel(0)
    sel = np.unique(np.concatenate([np.nonzero((eidx == 2).any(axis=1))[0], [0, T - 1], rng.choice(T, 24, replace=False)]))
    want = kqo.moe_ffn(tgu, tdn, X[sel], gp, up, dp, eidx[sel], ew[sel], H, I)
    rms = float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))
    assert np.all(np.abs(got[sel] - want) <= 1e-3 * rms + 1e-3 * np.abs(want))
    assert np.abs(got - tile).max() <= 1e-4 * rms + 1e-4 * np.abs(tile).max()


@pytest.mark.parametrize("inter,cap", [(512, 32), (1024, 48), (768, 64)])
@pytest.mark.parametrize("tgu,tdn", [(Q4_K, Q6_K), (Q5_K, Q4_K), (Q6_K, Q5_K)])
def test_moe_ffn_records_of_every_fill(gpu, kqo, tgu, tdn, inter, cap):  # noqa: F811
    """A workgroup walks the tiles of 16 pairs that its record fills: last records of one pair, of a tile less one, a tile, a tile
    and one more, up to the whole record.  Every token against its expert's matvec in 64 bits."""
    from backpack_amd import capi, kquant
    H = 512
    left = [n for t in range(0, cap, 16) for n in (t + 1, t + 15, t + 16)]
    whole = {32: 8, 48: 2, 64: 2}[cap]          # full records beside each: enough pairs that records of this size are chosen
    counts = np.array([whole * cap + n for n in left])
    E, k = len(counts), 2
    counts[0] += counts.sum() % k
    print("records of every fill", tgu, tdn, inter, cap, counts.sum(), flush=True)
    raw_g, _, gw = gpu.make_weight(tgu, E * inter, H, seed=51)
    raw_u, _, uw = gpu.make_weight(tgu, E * inter, H, seed=52)
    raw_d, _, dw = gpu.make_weight(tdn, E * H, inter, seed=53)
    rng = np.random.default_rng(cap)
    T = int(counts.sum()) // k
    eidx = np.repeat(np.arange(E, dtype=np.uint32), counts).reshape(k, T).T.copy()
    ew = rng.random((T, k)).astype(np.float32)
    X = (rng.standard_normal((T, H)) * 0.1).astype(np.float32)
    got = kquant.moe_ffn(gpu.dev(X), gw, uw, dw, gpu.dev(eidx.view(np.int32)), gpu.dev(ew), E).cpu().numpy()
    assert capi.last_form() == f"records_{cap}"
    want = np.zeros((T, H))
    for e in range(E):
        t, s = np.nonzero(eidx == e)
        x = X[t].astype(np.float64)
        g = x @ kqo.dequant(tgu, raw_g[e * inter:(e + 1) * inter], inter, H).astype(np.float64).T
        u = x @ kqo.dequant(tgu, raw_u[e * inter:(e + 1) * inter], inter, H).astype(np.float64).T
        y = (g / (1 + np.exp(-g)) * u) @ kqo.dequant(tdn, raw_d[e * H:(e + 1) * H], H, inter).astype(np.float64).T
        np.add.at(want, t, ew[t, s, None] * y)
    rms = float(np.sqrt(np.mean(want ** 2)))
    # two products of 22-bit splits one after the other, fp32 sums, an expf
    assert np.abs(got - want).max() <= 2.0 ** -15 * rms, float(np.abs(got - want).max()) / rms


@pytest.mark.parametrize("family", [0, 6])
def test_moe_ffn_pair_without_an_expert_adds_nothing(gpu, kqo, family):  # noqa: F811
    """Where pairs are grouped, one whose id is no expert's is dropped: its token gets the sum over its other slots,
    whatever the scratch memory held."""
    import torch
    from backpack_amd import capi
    T, E, k, H, I = 9, 4, 2, 512, 256
    _, gp, gw = gpu.make_weight(Q4_K, E * I, H, seed=84)
    _, up, uw = gpu.make_weight(Q4_K, E * I, H, seed=85)
    _, dp, dw = gpu.make_weight(Q6_K, E * H, I, seed=86)
    rng = np.random.default_rng(87)
    eidx = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.uint32)
    ew = rng.random((T, k)).astype(np.float32)
    X = (rng.standard_normal((T, H)) * 0.1).astype(np.float32)
    ew_known = ew.copy()
    want_idx = eidx.copy()
    for t, s in ((0, 0), (4, 1), (8, 0)):
        eidx[t, s], ew_known[t, s] = E + t, 0.0
    L = capi.lib()
    n = L.bpk_kq_moe_ffn_scratch_bytes(T, k, H, I)
    scratch = torch.full((n,), 0xFF, dtype=torch.uint8, device="cuda")     # every float a NaN
    out = torch.empty((T, H), dtype=torch.float32, device="cuda")
    x, idx, wt = gpu.dev(X), gpu.dev(eidx.view(np.int32)), gpu.dev(ew)
    capi.force_kernel(family)
    try:
        capi.check(L.bpk_kq_moe_ffn(Q4_K, Q6_K, x.data_ptr(), gw.data.data_ptr(), uw.data.data_ptr(), dw.data.data_ptr(), idx.data_ptr(),
                                    wt.data_ptr(), out.data_ptr(), T, k, E, H, I, scratch.data_ptr(), n, None))
    finally:
        capi.force_kernel(0)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    want = kqo.moe_ffn(Q4_K, Q6_K, X, gp, up, dp, want_idx, ew_known, H, I)
    rms = float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))
    assert np.all(np.abs(got - want) <= 1e-3 * rms + 1e-3 * np.abs(want))


@pytest.mark.parametrize("type_", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("M,N,K", [(1, 1, 256), (17, 255, 512), (33, 257, 2816), (100, 520, 4096), (128, 256, 256), (129, 300, 1024),
                                   (257, 513, 4096), (300, 256, 4352), (512, 300, 4096)])
def test_short_prompt_vs_oracle(gpu, kqo, type_, M, N, K):  # noqa: F811
    """bf16 rows of a short prompt: tokens around the groups of 16 and 128 (three and four groups too), rows around 256, K cut over workgroups and
    not, with a bias; against the oracle on the same bf16 rows and against the GEMM's 128-tile (the same products)."""
    import torch
    from backpack_amd import capi, kquant
    print("short", type_, M, N, K, flush=True)
    raw, packed, w = gpu.make_weight(type_, N, K, seed=M + N)
    rng = np.random.default_rng(K + M)
    X = gpu.dev(rng.standard_normal((M, K)).astype(np.float32)).bfloat16()
    bias = gpu.dev(rng.standard_normal(N).astype(np.float32))
    capi.force_kernel(9)
    try:
        got = kquant.matmul(X, w, bias=bias).cpu().numpy()
    finally:
        capi.force_kernel(0)
    assert (capi.last_kernel(), capi.last_form()) == ("gemm_bf16", "short_prompt")
    capi.set_option("gemm_tile", 128)
    try:
        gemm = kquant.matmul(X, w, bias=bias).cpu().numpy()
        assert (capi.last_kernel(), capi.last_form()) == ("gemm_bf16", "")
    finally:
        capi.set_option("gemm_tile", 0)
    want = kqo.matmul(type_, X.float().cpu().numpy(), packed, N, K) + bias.cpu().numpy()
    rms = float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))
    # weights rounded to bf16: 2^-9 per product, K independent ones
    assert np.sqrt(np.mean((got - want) ** 2.0)) <= 2.0 ** -8 * rms
    # the same products in another order: fp32 sums of K of them
    assert np.abs(got - gemm).max() <= 2.0 ** -23 * K ** 0.5 * 8 * max(rms, float(np.abs(want).max()))


@pytest.mark.parametrize("type_", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("M", [32, 48, 63, 80, 81, 112, 113])
@pytest.mark.parametrize("N,blocks", [(271, 1), (40, 2), (9, 3), (257, 18)])
def test_short_prompt_tiles_and_walks(gpu, kqo, type_, M, N, blocks):  # noqa: F811
    """Every number of token tiles (odd ones, where half the waves have a load less), walks of one superblock and two (K is cut into
    single ones on rows this short; three blocks of nine Q4_K rows are one walk of three at 32 tokens), fewer rows than a tile; against
    64-bit sums of the bf16 weights."""
    import torch
    from backpack_amd import capi, kquant
    K = 256 * blocks
    raw, _, w = gpu.make_weight(type_, N, K, seed=M + N)
    rng = np.random.default_rng(K + M)
    X = gpu.dev(rng.standard_normal((M, K)).astype(np.float32)).bfloat16()
    capi.force_kernel(9)
    try:
        got = kquant.matmul(X, w).cpu().numpy()
        again = kquant.matmul(X, w).cpu().numpy()
    finally:
        capi.force_kernel(0)
    assert capi.last_form() == "short_prompt" and np.array_equal(got, again)
    wb = torch.from_numpy(kqo.dequant(type_, raw, N, K)).bfloat16().double().numpy()
    want = X.double().cpu().numpy() @ wb.T
    rms = float(np.sqrt(np.mean(want ** 2)))
    # fp32 sums of K products
    assert np.abs(got - want).max() <= 2.0 ** -23 * K ** 0.5 * 8 * max(rms, float(np.abs(want).max()))


@pytest.mark.parametrize("N,blocks", [(20000, 10), (30001, 7)])
@pytest.mark.parametrize("type_", [Q4_K, Q5_K, Q6_K])
def test_short_prompt_long_walks(gpu, kqo, type_, N, blocks):  # noqa: F811
    """Walks of four superblocks and more, in which the ring comes back to where it began and a superblock's loads are sent two steps
    ahead of it, at odd and even numbers of token tiles: whole outputs against the GEMM, which has the same products, rows of the first,
    of inner and of the last tiles against 64-bit sums."""
    import torch
    from backpack_amd import capi, kquant
    K = 256 * blocks
    raw, _, w = gpu.make_weight(type_, N, K, seed=blocks)
    at = np.r_[0:17, 255:257, 8191:8193, N - 33:N]
    wb = torch.from_numpy(kqo.dequant(type_, raw[at], len(at), K)).bfloat16().double().numpy()
    for M in (17, 48, 64, 80, 96, 100, 113):
        print("short, long walk", type_, M, N, K, flush=True)
        _, tokens, splits = capi.short_plan(type_, M, N, K)
        assert tokens == max(32, -(-M // 16) * 16) and -(-blocks // splits) >= 4, (tokens, splits)
        X = gpu.dev(np.random.default_rng(M).standard_normal((M, K)).astype(np.float32)).bfloat16()
        capi.force_kernel(9)
        try:
            got = kquant.matmul(X, w)
        finally:
            capi.force_kernel(0)
        assert capi.last_form() == "short_prompt"
        capi.set_option("gemm_tile", 128)
        try:
            gemm = kquant.matmul(X, w)
        finally:
            capi.set_option("gemm_tile", 0)
        want = X.double().cpu().numpy() @ wb.T
        # fp32 sums of K products, once and in two orders
        bound = 2.0 ** -23 * K ** 0.5 * 8
        assert np.abs(got[:, at].cpu().numpy() - want).max() <= bound * float(np.abs(want).max())
        assert float((got - gemm).abs().max()) <= 2 * bound * float(gemm.abs().max())


def test_forced_families_run_what_they_name(gpu):  # noqa: F811
    """Family 4 on bf16 X is the tiled GEMM and 9 the short-prompt kernel, whatever the price says; families that have
    no form of a call refuse it instead of answering from another kernel."""
    import torch
    from backpack_amd import capi, kquant
    type_, M, N, K = Q4_K, 100, 520, 4096
    raw, packed, w = gpu.make_weight(type_, N, K, seed=3)
    x32 = gpu.dev(np.random.default_rng(3).standard_normal((M, K)).astype(np.float32))
    X = x32.bfloat16()
    auto = kquant.matmul(X, w)
    plan = capi.gemm_plan(type_, M, N, K)                  # the GEMM's own choice: equal shares of the 256-tiles
    capi.set_option("gemm_tile", 256)
    capi.set_option("gemm_split", 2)
    try:
        assert capi.gemm_plan(type_, M, N, K) == plan
        tile = kquant.matmul(X, w)
    finally:
        capi.set_option("gemm_tile", 0)
        capi.set_option("gemm_split", 0)
    assert not torch.equal(auto, tile)                     # priced below the GEMM: K cut over workgroups
    raw2, packed2, we = gpu.make_weight(type_, 4 * 256, 256, seed=4)
    eidx = torch.zeros((3, 1), dtype=torch.int32, device="cuda")
    try:
        capi.force_kernel(4)
        assert torch.equal(kquant.matmul(X, w), tile)
        capi.force_kernel(9)
        assert torch.equal(kquant.matmul(X, w), auto)

        def refused(call):
            with pytest.raises(capi.BpkError) as e:
                call()
            assert e.value.code == -2
        refused(lambda: kquant.matmul(x32, w))
        refused(lambda: kquant.matmul(X.repeat(6, 1), w))  # 600 tokens
        for family in (8, 9):
            capi.force_kernel(family)
            refused(lambda: kquant.moe_matmul(x32[:3, :256].contiguous(), we, eidx, 4))
            # one slot per token: the split X does not fit beside the records
            refused(lambda: kquant.moe_ffn(x32[:3, :256].contiguous(), we, we, we, eidx, torch.ones((3, 1), device="cuda"), 4))
    finally:
        capi.force_kernel(0)


@pytest.mark.parametrize("type_,M,N,K,form", [
    # one chunk of X per workgroup of the tile kernel, one round of the CUs, Q6_K: the tile kernel
    (Q6_K, 17, 2048, 512, ""), (Q6_K, 32, 4096, 1024, ""), (Q6_K, 24, 512, 14336, ""), (Q6_K, 32, 768, 8448, ""),
    # one superblock, more chunks, more rows, more tokens, other types: the many-token kernel
    (Q6_K, 17, 2048, 256, "many_token"), (Q6_K, 17, 2048, 1280, "many_token"), (Q6_K, 17, 4097, 1024, "many_token"),
    (Q6_K, 33, 2048, 1024, "many_token"), (Q6_K, 17, 256, 8448, "many_token"), (Q6_K, 17, 769, 16384, "many_token"),
    (Q6_K, 17, 512, 16640, "many_token"), (Q4_K, 17, 2048, 1024, "many_token"), (Q5_K, 17, 2048, 1024, "many_token")])
def test_dispatch_of_17_to_32_tokens(gpu, kqo, type_, M, N, K, form):  # noqa: F811
    """Small Q6_K matrices stay on the 16-token tiles, where those are the faster; the same outputs as that kernel forced,
    and the many-token kernel on the same call."""
    import torch
    from backpack_amd import capi, kquant
    raw, packed, w = gpu.make_weight(type_, N, K, seed=M + K)
    x = np.random.default_rng(N).standard_normal((M, K)).astype(np.float32)
    X = gpu.dev(x)
    got = kquant.matmul(X, w)
    assert (capi.last_kernel(), capi.last_form()) == ("mtile", form)
    try:
        capi.force_kernel(8 if form else 6)
        assert torch.equal(got, kquant.matmul(X, w))
        capi.force_kernel(6 if form else 8)
        other = kquant.matmul(X, w).cpu().numpy()
    finally:
        capi.force_kernel(0)
    cols = np.arange(0, N, max(1, N // 64))                  # (the oracle on some of the rows)
    part = packed.reshape(N, -1)[cols].reshape(-1)
    for y in (got.cpu().numpy(), other):
        gpu.check_matmul(kqo, type_, np.ascontiguousarray(y[:, cols]), x, part, len(cols), K, label="dispatch", slack=2e-5)


@pytest.mark.parametrize("M,pro,res,epi,form", [(24, 1, False, 0, ""), (17, 0, True, 0, ""), (17, 0, False, 2, ""), (24, 1, False, 2, "many_token"),
                                                (17, 2, True, 0, "many_token"), (25, 0, True, 0, "many_token")])
def test_dispatch_of_17_to_32_fused_tokens(gpu, M, pro, res, epi, form):  # noqa: F811
    """A fused call that saves the many-token kernel one launch stays on the tile kernel up to 24 tokens."""
    from backpack_amd import capi, kquant
    N, K = 512, 1024
    raw, packed, w = gpu.make_weight(Q6_K, 2 * N if epi else N, K, seed=M)
    rng = np.random.default_rng(M)
    x = gpu.dev(rng.standard_normal((M, 2 * K if pro == 2 else K)).astype(np.float32))
    nw = gpu.dev(rng.standard_normal(K).astype(np.float32)) if pro == 1 else None
    r = gpu.dev(rng.standard_normal((M, N)).astype(np.float32)) if res else None
    args = dict(norm_w=nw, eps=1e-5, residual=r, epilogue=epi)
    got = kquant.matmul_fused(x, w, pro, **args).cpu().numpy()
    assert capi.last_form() == form
    try:
        capi.force_kernel(8)
        other = kquant.matmul_fused(x, w, pro, **args).cpu().numpy()
        assert capi.last_form() == "many_token"
    finally:
        capi.force_kernel(0)
    rms = float(np.sqrt(np.mean(other.astype(np.float64) ** 2)))
    # both split x into 22 bits of its superblock's largest; the tile kernel adds 2 x 32 products per matrix instruction chain
    assert float(np.abs(got - other).max()) <= 5e-5 * rms + 1e-5 * float(np.abs(other).max())


@pytest.mark.parametrize("tgu,tdn,E,k,T,H,I,form", [
    # few workgroups and a long walk: the tile kernel
    (Q6_K, Q6_K, 8, 2, 12, 2048, 256, ""), (Q6_K, Q4_K, 8, 2, 40, 1280, 512, ""), (Q6_K, Q6_K, 8, 2, 5, 1024, 512, ""), (Q5_K, Q6_K, 8, 2, 8, 1536, 768, ""),
    (Q4_K, Q6_K, 8, 2, 8, 1280, 1024, ""),
    # Q4_K down; from four pairs per expert on; hidden of one chunk; more experts
    (Q4_K, Q4_K, 8, 2, 8, 2048, 512, "records_16"), (Q5_K, Q6_K, 8, 2, 16, 1536, 768, "records_16"), (Q6_K, Q6_K, 8, 2, 16, 1024, 512, "records_16"),
    (Q6_K, Q6_K, 64, 4, 40, 1280, 512, "records_16")])
def test_dispatch_of_expert_layers_with_few_workgroups(gpu, kqo, tgu, tdn, E, k, T, H, I, form):  # noqa: F811
    from backpack_amd import capi, kquant
    _, gp, gw = gpu.make_weight(tgu, E * I, H, seed=91)
    _, up, uw = gpu.make_weight(tgu, E * I, H, seed=92)
    _, dp, dw = gpu.make_weight(tdn, E * H, I, seed=93)
    rng = np.random.default_rng(T)
    eidx = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.uint32)
    ew = rng.random((T, k)).astype(np.float32)
    X = (rng.standard_normal((T, H)) * 0.1).astype(np.float32)
    args = (gpu.dev(X), gw, uw, dw, gpu.dev(eidx.view(np.int32)), gpu.dev(ew), E)
    got = kquant.moe_ffn(*args).cpu().numpy()
    assert (capi.last_kernel(), capi.last_form()) == ("moe_ffn_mtile", form)
    capi.force_kernel(8 if form else 6)
    try:
        assert np.array_equal(got, kquant.moe_ffn(*args).cpu().numpy())
    finally:
        capi.force_kernel(0)
    want = kqo.moe_ffn(tgu, tdn, X, gp, up, dp, eidx, ew, H, I)
    rms = float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))
    assert np.all(np.abs(got - want) <= 1e-3 * rms + 1e-3 * np.abs(want))


@pytest.mark.parametrize("extra", [0, 1, 40])
def test_moe_records_around_a_round(gpu, kqo, extra):  # noqa: F811
    """64 records, or a few more: the number of row groups that a workgroup walks is chosen on the device from the records'
    number.  Gate and up have 14 groups: four each at 64 records (64 x 4 workgroups are a round of 256 CUs, the last of a
    record's walks two), five from 65 on, seven at 104.  Some tokens in 64 bits, all against the 16-token tile kernel."""
    from backpack_amd import capi, kquant
    E, k, H, I, cap = 64, 2, 512, 1792, 32
    raw_g, _, gw = gpu.make_weight(Q4_K, E * I, H, seed=41)
    raw_u, _, uw = gpu.make_weight(Q4_K, E * I, H, seed=42)
    raw_d, _, dw = gpu.make_weight(Q6_K, E * H, I, seed=43)
    rng = np.random.default_rng(extra)
    counts = np.array([33] * extra + [24] * (E - extra))            # 33 pairs take two records
    counts[-1] += counts.sum() % k
    eidx = np.repeat(np.arange(E, dtype=np.uint32), counts)
    T = len(eidx) // k
    eidx = eidx.reshape(k, T).T.copy()
    records = int(sum((c + cap - 1) // cap for c in np.bincount(eidx.reshape(-1), minlength=E)))
    assert records == 64 + extra
    ew = rng.random((T, k)).astype(np.float32)
    X = (rng.standard_normal((T, H)) * 0.1).astype(np.float32)
    args = (gpu.dev(X), gw, uw, dw, gpu.dev(eidx.view(np.int32)), gpu.dev(ew), E)
    got = kquant.moe_ffn(*args).cpu().numpy()
    assert capi.last_form() == f"records_{cap}"
    capi.force_kernel(6)
    try:
        tile = kquant.moe_ffn(*args).cpu().numpy()
    finally:
        capi.force_kernel(0)
    rms = float(np.sqrt(np.mean(tile.astype(np.float64) ** 2)))
    assert np.abs(got - tile).max() <= 1e-4 * rms + 1e-4 * np.abs(tile).max()
    for t in rng.choice(T, 12, replace=False):
        want = np.zeros(H)
        for s in range(k):
            e = int(eidx[t, s])
            g = kqo.dequant(Q4_K, raw_g[e * I:(e + 1) * I], I, H).astype(np.float64) @ X[t]
            u = kqo.dequant(Q4_K, raw_u[e * I:(e + 1) * I], I, H).astype(np.float64) @ X[t]
            want += float(ew[t, s]) * (kqo.dequant(Q6_K, raw_d[e * H:(e + 1) * H], H, I).astype(np.float64) @ (g / (1 + np.exp(-g)) * u))
        # two products of 22-bit splits one after the other, fp32 sums, an expf
        assert np.abs(got[t] - want).max() <= 2.0 ** -15 * rms, float(np.abs(got[t] - want).max()) / rms


@pytest.mark.parametrize("type_,M,N,K,form", [(Q6_K, 3, 128256, 256, "many_token"), (Q6_K, 8, 61500, 1024, "many_token"), (Q4_K, 5, 128257, 512, "many_token"),
                                              (Q5_K, 8, 131072, 256, "many_token"), (Q4_K, 8, 61500, 1024, ""), (Q5_K, 4, 80000, 512, "")])
def test_few_tokens_on_many_rows(gpu, kqo, type_, M, N, K, form):  # noqa: F811
    """3 to 8 tokens on matrices whose rows fill the CUs: the many-token kernel where its rounds come out, else the tiles.
    Windows of rows against the oracle."""
    from backpack_amd import capi, kquant, synth
    print("few tokens", type_, M, N, K, flush=True)
    raw, packed, w = gpu.make_weight(type_, N, K, seed=M)
    X = np.random.default_rng(N).standard_normal((M, K)).astype(np.float32)
    got = kquant.matmul(gpu.dev(X), w).cpu().numpy()
    assert (capi.last_kernel(), capi.last_form()) == ("mtile", form)
    words = synth.row_stride_words(type_, K)
    for a, b in ((0, 270), (N // 2, N // 2 + 300), (N - 270, N)):
        gpu.check_matmul(kqo, type_, np.ascontiguousarray(got[:, a:b]), X, packed[a * words:b * words], b - a, K, label="few tokens", slack=1e-5)


def test_header_names_the_smallest_call_that_uses_the_shared_scratch(gpu):  # noqa: F811
    """The many-token kernel's split X lies in scratch that calls share: from the number of tokens that the header's list gives,
    on the matrices it takes first (many rows), and from no smaller one."""
    import os
    from backpack_amd import capi, kquant
    header = open(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "bpk_kquant.h")).read()
    assert "any of three tokens and more" in " ".join(header.replace("\n *", " ").split())
    N, K = 128256, 256
    raw, packed, w = gpu.make_weight(Q6_K, N, K, seed=1)
    for M, form in ((1, ""), (2, ""), (3, "many_token")):
        kquant.matmul(gpu.dev(np.ones((M, K), np.float32)), w)
        assert capi.last_form() == form, M


@pytest.mark.parametrize("type_,M", [(Q4_K, 17), (Q6_K, 17), (Q4_K, 5)])
def test_rows_farther_apart_than_32_bit_offsets_reach(gpu, kqo, type_, M):  # noqa: F811
    """Rows 302 MB apart: a tile of sixteen spans more than 2^32 bytes.  The kernels that hold a row's place in 32 bits leave such a
    call to one that does not."""
    import torch
    from backpack_amd import capi, kquant, synth
    N, K, stride = 17, 256, 0x12000000
    print("far rows", type_, M, flush=True)
    raw, packed, w = gpu.make_weight(type_, N, K, seed=9)
    row = synth.row_stride_words(type_, K) * 4
    data = torch.zeros(N * stride + 16, dtype=torch.uint8, device="cuda")
    body = torch.from_numpy(packed.view(np.uint8).reshape(N, row)).cuda()
    for n in range(N):
        data[n * stride:n * stride + row] = body[n]
    far = kquant.KQuantPacked(data, type_, N, K, stride // 4, 1)
    X = np.random.default_rng(M).standard_normal((M, K)).astype(np.float32)
    got = kquant.matmul(gpu.dev(X), far).cpu().numpy()
    gpu.check_matmul(kqo, type_, got, X, packed, N, K, label="far rows", slack=1e-5)
    for family in (6, 8):
        capi.force_kernel(family)
        try:
            with pytest.raises(capi.BpkError) as e:
                kquant.matmul(gpu.dev(X), far)
            assert e.value.code == -2
        finally:
            capi.force_kernel(0)
    del data, far
    torch.cuda.empty_cache()


@pytest.mark.parametrize("type_", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("M,blocks", [(1, 1), (16, 1), (9, 2), (16, 3), (16, 4), (16, 6)])
def test_walks_of_few_superblocks_at_16_tokens(gpu, kqo, type_, M, blocks):  # noqa: F811
    """Nothing is requested past the end of the walk: every place in the ring as the last one, K in one piece and cut into walks of
    one superblock."""
    from backpack_amd import capi, kquant
    N, K = 270, 256 * blocks
    raw, packed, w = gpu.make_weight(type_, N, K, seed=blocks)
    X = np.random.default_rng(M).standard_normal((M, K)).astype(np.float32)
    capi.force_kernel(8)
    try:
        for splits in (1, blocks):
            capi.set_option("gemv_splits", splits)
            got = kquant.matmul(gpu.dev(X), w).cpu().numpy()
            assert capi.last_form() == "many_token"
            gpu.check_matmul(kqo, type_, got, X, packed, N, K, label="walk", slack=1e-5)
    finally:
        capi.force_kernel(0)
        capi.set_option("gemv_splits", 0)


@pytest.mark.parametrize("type_,M,N,K", [(Q4_K, 9, 256 * 601 + 3, 256), (Q5_K, 16, 256 * 513 + 1, 512), (Q6_K, 12, 256 * 767, 256)])
def test_three_row_groups_per_workgroup_at_16_tokens(gpu, kqo, type_, M, N, K):  # noqa: F811
    """Between two and three rounds of 256 rows per CU: workgroups of three groups, the last one ragged.  Windows of rows around the
    workgroups' borders against the oracle."""
    from backpack_amd import capi, kquant, synth
    print("three groups", type_, M, N, K, flush=True)
    raw, packed, w = gpu.make_weight(type_, N, K, seed=M)
    X = np.random.default_rng(N).standard_normal((M, K)).astype(np.float32)
    got = kquant.matmul(gpu.dev(X), w).cpu().numpy()
    assert (capi.last_kernel(), capi.last_form()) == ("mtile", "many_token")
    words = synth.row_stride_words(type_, K)
    for a, b in ((0, 300), (768 * 100 - 20, 768 * 100 + 300), (N - 900, N)):
        gpu.check_matmul(kqo, type_, np.ascontiguousarray(got[:, a:b]), X, packed[a * words:b * words], b - a, K, label="three groups", slack=1e-5)


@pytest.mark.parametrize("k", [8, 9, 11])
def test_moe_ffn_of_more_than_eight_slots(gpu, kqo, k):  # noqa: F811
    """The sum over a token's slots takes them eight at a time: exactly eight, one and three more."""
    from backpack_amd import capi, kquant
    T, E, H, I = 30, 16, 768, 256
    print("slots", k, flush=True)
    _, gp, gw = gpu.make_weight(Q4_K, E * I, H, seed=61)
    _, up, uw = gpu.make_weight(Q4_K, E * I, H, seed=62)
    _, dp, dw = gpu.make_weight(Q5_K, E * H, I, seed=63)
    rng = np.random.default_rng(k)
    eidx = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.uint32)
    ew = rng.random((T, k)).astype(np.float32)
    X = (rng.standard_normal((T, H)) * 0.1).astype(np.float32)
    got = kquant.moe_ffn(gpu.dev(X), gw, uw, dw, gpu.dev(eidx.view(np.int32)), gpu.dev(ew), E).cpu().numpy()
    assert capi.last_form().startswith("records_")
    want = kqo.moe_ffn(Q4_K, Q5_K, X, gp, up, dp, eidx, ew, H, I)
    rms = float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))
    # (a slot left out or counted twice is off by a third of the rms)
    assert np.all(np.abs(got - want) <= 1e-3 * rms + 1e-3 * np.abs(want))


def _q6_of_the_whole_range(gpu, N, K, seed):
    """A Q6_K matrix with scales over the whole of int8 and quants over all 64 values: (packed, w, exact weights, weights with
    scale * (q - 32) rounded to fp16, as a kernel without the third product would multiply them)."""
    from backpack_amd import kquant, synth
    rng = np.random.default_rng(seed)
    d, _, q = synth.q6k_fields(rng, N, K // 256)
    sc = rng.integers(-128, 128, size=(N, K // 256, 16), dtype=np.int8)
    sc[:, :, 0], sc[:, :, 5] = -128, 127                      # (products of up to 13 bits: 128 * 32)
    q.reshape(-1)[::97] = 0
    packed = synth.pack_rows(synth.Q6_K, synth.q6k_encode(d, sc, q).reshape(N, -1), N, K)
    exact = synth.q6k_decode_f64(d, sc, q)
    dd = np.repeat(d.astype(np.float64).reshape(N, -1), 256, axis=1)
    dd[dd == 0.0] = 1.0
    coarse = (exact / dd).astype(np.float16).astype(np.float64) * dd
    return packed, kquant.upload(synth.Q6_K, packed, N, K), exact, coarse


# tiles of 16 tokens one to four; few tokens on many rows (by itself); K cut into walks of a superblock and in one piece
@pytest.mark.parametrize("M,N,K,splits", [(16, 257, 1280, 0), (17, 300, 512, 1), (33, 270, 1024, 0), (64, 256, 768, 1), (100, 130, 2816, 0), (5, 61500, 512, 0)])
def test_q6_scales_of_the_whole_range(gpu, kqo, M, N, K, splits):  # noqa: F811
    """Beyond 2048 scale * (q - 32) needs the third product: against 64 bits, with a limit that weights rounded to fp16 exceed."""
    from backpack_amd import capi, kquant
    print("q6 range", M, N, K, splits, flush=True)
    packed, w, exact, coarse = _q6_of_the_whole_range(gpu, N, K, seed=M)
    X = np.random.default_rng(K).standard_normal((M, K)).astype(np.float32)
    if M > 8:
        capi.force_kernel(8)
    capi.set_option("gemv_splits", splits)
    try:
        got = kquant.matmul(gpu.dev(X), w).cpu().numpy()
    finally:
        capi.force_kernel(0)
        capi.set_option("gemv_splits", 0)
    assert capi.last_form() == "many_token"
    want, bad = X.astype(np.float64) @ exact.T, X.astype(np.float64) @ coarse.T
    rms = float(np.sqrt(np.mean(want ** 2)))
    # x keeps 22 bits of its superblock's largest, lo * Wl (2^-22 of a product) is dropped, sums in fp32 over chains of up to 8 + K / 256
    # instructions: 2^-17 of the rms is above all of them together
    limit = 2.0 ** -17 * rms
    assert float(np.abs(got - want).max()) <= limit, float(np.abs(got - want).max()) / rms
    assert float(np.abs(bad - want).max()) > 20 * limit


@pytest.mark.parametrize("T,cap", [(30, 16), (700, 32), (1300, 48)])
def test_moe_ffn_q6_scales_of_the_whole_range(gpu, T, cap):  # noqa: F811
    """The same in both launches of an expert layer, on records of 16 and of more pairs, against 64 bits."""
    from backpack_amd import capi, kquant
    E, k, H, I = 4, 2, 512, 512
    print("moe q6 range", T, flush=True)
    _, gw, g64, g16 = _q6_of_the_whole_range(gpu, E * I, H, 1)
    _, uw, u64, u16 = _q6_of_the_whole_range(gpu, E * I, H, 2)
    _, dw, d64, d16 = _q6_of_the_whole_range(gpu, E * H, I, 3)
    rng = np.random.default_rng(T)
    eidx = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.uint32)
    ew = rng.random((T, k)).astype(np.float32)
    X = (rng.standard_normal((T, H)) * 0.01).astype(np.float32)
    got = kquant.moe_ffn(gpu.dev(X), gw, uw, dw, gpu.dev(eidx.view(np.int32)), gpu.dev(ew), E).cpu().numpy()
    assert capi.last_form() == f"records_{cap}"

    def layer(g, u, d):
        out = np.zeros((T, H))
        for e in range(E):
            t, s = np.nonzero(eidx == e)
            x = X[t].astype(np.float64)
            gate, up = x @ g[e * I:(e + 1) * I].T, x @ u[e * I:(e + 1) * I].T
            np.add.at(out, t, ew[t, s].astype(np.float64)[:, None] * ((gate / (1 + np.exp(-gate)) * up) @ d[e * H:(e + 1) * H].T))
        return out
    want = layer(g64, u64, d64)
    rms = float(np.sqrt(np.mean(want ** 2)))
    # two products as above one after the other, gate's error through silu (slope up to 1.1, beside |gate| of the rms's size) and expf's
    limit = 2.0 ** -16 * rms
    assert float(np.abs(got - want).max()) <= limit, float(np.abs(got - want).max()) / rms
    for planted in (layer(g16, u16, d64), layer(g64, u64, d16)):
        assert float(np.abs(planted - want).max()) > 5 * limit


@pytest.mark.parametrize("grid", [8, 24, 4096])
def test_moe_records_in_a_second_dimension_of_the_grid(gpu, grid):  # noqa: F811
    """What a launch of more than 2^22 workgroups over records does, at a size that a test can afford: the same outputs, bit for
    bit, with the first dimension held to a few workgroups."""
    from backpack_amd import capi, kquant
    E, k, H, I = 6, 2, 512, 768
    _, gp, gw = gpu.make_weight(Q4_K, E * I, H, seed=51)
    _, up, uw = gpu.make_weight(Q4_K, E * I, H, seed=52)
    _, dp, dw = gpu.make_weight(Q6_K, E * H, I, seed=53)
    for T in (37, 400):
        rng = np.random.default_rng(T)
        eidx = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.uint32)
        args = (gpu.dev((rng.standard_normal((T, H)) * 0.1).astype(np.float32)), gw, uw, dw, gpu.dev(eidx.view(np.int32)), gpu.dev(rng.random((T, k)).astype(np.float32)), E)
        want = kquant.moe_ffn(*args).cpu().numpy()
        assert capi.last_form().startswith("records_")
        capi.set_option("moe_grid", grid)
        try:
            got = kquant.moe_ffn(*args).cpu().numpy()
        finally:
            capi.set_option("moe_grid", 0)
        assert np.array_equal(got, want)
    with pytest.raises(capi.BpkError):
        capi.set_option("moe_grid", 12)      # not a multiple of the XCDs


@pytest.mark.parametrize("type_,M,N,K,pro,epi,res,form", [
    (Q4_K, 16, 28672, 4096, 1, 2, False, "many_token"), (Q6_K, 16, 4096, 14336, 0, 0, True, "many_token"), (Q6_K, 9, 4096, 14336, 0, 0, True, "many_token"),
    (Q4_K, 16, 4096, 4096, 0, 0, True, None), (Q4_K, 8, 6144, 4096, 1, 0, False, None), (Q5_K, 12, 36896, 1024, 1, 3, False, "many_token"),
    (Q6_K, 13, 35999, 1024, 0, 0, False, "many_token"), (Q5_K, 13, 20817, 4608, 0, 0, False, "many_token"), (Q4_K, 5, 700, 512, 1, 0, True, None)])
def test_dispatch_of_5_to_16_tokens(gpu, type_, M, N, K, pro, epi, res, form):  # noqa: F811
    """The many-token kernel where it is priced below the tiles, both ways the same function: against the tile kernel, which splits x
    into the same 22 bits; without a workspace a fused call stays one launch."""
    import torch
    from backpack_amd import capi, kquant
    print("5 to 16 tokens", type_, M, N, K, pro, epi, res, flush=True)
    _, _, w = gpu.make_weight(type_, N, K, seed=M)
    rng = np.random.default_rng(N)
    X = gpu.dev(rng.standard_normal((M, K)).astype(np.float32))
    nw = gpu.dev((1 + 0.1 * rng.standard_normal(K)).astype(np.float32)) if pro == 1 else None
    R = gpu.dev(rng.standard_normal((M, N)).astype(np.float32)) if res else None
    fused = pro or epi or res

    def call(**k):
        return kquant.matmul_fused(X, w, pro, norm_w=nw, eps=1e-5, residual=R, epilogue=epi, **k) if fused else kquant.matmul(X, w)
    got = call()
    assert (capi.last_kernel(), capi.last_form()) == (("mtile", form) if form or not fused else ("mtile_fused", ""))
    capi.force_kernel(6)
    try:
        tile = call()
    finally:
        capi.force_kernel(0)
    if fused:
        one = call(allow_workspace=False)
        assert capi.last_kernel() == "mtile_fused" and torch.equal(one, tile)
    if res:      # in place
        y = R.clone()
        kquant.matmul_fused(X, w, pro, norm_w=nw, eps=1e-5, residual=y, out=y)
        assert torch.equal(y, got)
    # splits of x into 22 bits and fp32 sums in two orders; an activation multiplies two such: 1e-5 apart at most over 150000 random calls
    assert float((got - tile).double().norm() / tile.double().norm()) <= 2e-5


# rows of W, us on one MI355X: the launches of prologue, product and epilogue, the many-token kernel with all of it inside
@pytest.mark.parametrize("type_,M,rows,K,pro,epi,separate_us,wide_us", [
    (Q6_K, 12, 32776, 256, 0, 2, 25.2, 9.5), (Q4_K, 15, 7182, 256, 1, 3, 17.5, 8.2), (Q6_K, 16, 1864, 11008, 1, 2, 44.6, 22.4),
    (Q4_K, 8, 1954, 12032, 1, 3, 36.9, 18.0), (Q5_K, 16, 32770, 512, 1, 3, 21.6, 11.7),
    (Q5_K, 5, 696, 1024, 0, 2, 7.8, 14.1), (Q6_K, 8, 2066, 768, 1, 3, 10.7, 13.9), (Q4_K, 5, 812, 3072, 0, 3, 10.2, 11.9),
    # rows that fill the CUs
    (Q4_K, 9, 61202, 256, 1, 2, None, None), (Q6_K, 16, 61202, 512, 0, 2, None, None)])
def test_5_to_16_tokens_with_an_epilogue_over_any_rows(gpu, type_, M, rows, K, pro, epi, separate_us, wide_us):  # noqa: F811
    """The tile kernel's gate and up tiles need a multiple of 32 rows; other calls weigh the many-token kernel against what would run."""
    import torch
    from backpack_amd import capi, kquant
    print("epilogue, any rows", type_, M, rows, K, pro, epi, flush=True)
    _, _, w = gpu.make_weight(type_, rows, K, seed=M)
    rng = np.random.default_rng(rows)
    X = gpu.dev(rng.standard_normal((M, K)).astype(np.float32))
    nw = gpu.dev((1 + 0.1 * rng.standard_normal(K)).astype(np.float32)) if pro else None
    got = kquant.matmul_fused(X, w, pro, norm_w=nw, eps=1e-5, epilogue=epi)
    assert (capi.last_form() == "many_token") == (wide_us is None or wide_us < separate_us), (capi.last_kernel(), capi.last_form())
    capi.set_option("fused_separate", 1)
    try:
        want = kquant.matmul_fused(X, w, pro, norm_w=nw, eps=1e-5, epilogue=epi)
    finally:
        capi.set_option("fused_separate", 0)
    # splits of x into 22 bits and fp32 sums in two orders, in each of the two factors: 1e-5 apart at most over 150000 random calls
    assert float((got - want).double().norm() / want.double().norm()) <= 2e-5


@pytest.mark.parametrize("type_,M,N,wide", [(Q4_K, 9, 61185, True), (Q5_K, 16, 61185, True), (Q6_K, 7, 96678, True), (Q4_K, 5, 66000, False),
                                            (Q4_K, 9, 60928, False)])
def test_act_prologue_on_many_rows(gpu, type_, M, N, wide):  # noqa: F811
    """Behind an act * up prologue 5 to 16 tokens go by the rows as plain calls do, given a workspace; without one the call is the tile
    kernel's one launch."""
    import torch
    from backpack_amd import capi, kquant
    K = 256
    print("act prologue", type_, M, N, flush=True)
    _, _, w = gpu.make_weight(type_, N, K, seed=M)
    X = gpu.dev(np.random.default_rng(N).standard_normal((M, 2 * K)).astype(np.float32))
    got = kquant.matmul_fused(X, w, capi.PRO_SILU_MUL)
    assert (capi.last_form() == "many_token") == wide
    want = kquant.matmul_fused(X, w, capi.PRO_SILU_MUL, allow_workspace=False)
    assert capi.last_kernel() == "mtile_fused"
    assert float((got - want).double().norm() / want.double().norm()) <= 2e-5     # (as above)


# us on one MI355X, each kernel forced: the tile kernel, the many-token kernel
@pytest.mark.parametrize("type_,M,N,K,pro,res,tile_us,wide_us", [
    # few rows: a tile per workgroup; a workgroup whose tiles are not all there
    (Q6_K, 13, 41, 1024, 0, False, 7.1, 12.8), (Q6_K, 14, 64, 1024, 0, False, 7.3, 12.8), (Q4_K, 14, 47, 5888, 0, False, 11.2, 15.4),
    (Q5_K, 13, 43, 2048, 0, False, 11.3, 14.1), (Q4_K, 12, 64, 3584, 0, False, 10.5, 11.9), (Q6_K, 5, 44, 3840, 0, False, 12.2, 13.7),
    # short rows, many of them, a few tokens
    (Q6_K, 8, 31785, 512, 0, False, 9.4, 12.3), (Q6_K, 6, 29803, 512, 1, True, 10.4, 12.6),
    # the other side
    (Q6_K, 16, 33720, 256, 0, False, 24.4, 9.2), (Q6_K, 14, 34714, 256, 1, False, 25.3, 9.4), (Q6_K, 16, 47, 2048, 0, False, 15.4, 12.5),
    (Q6_K, 16, 40009, 256, 0, True, 25.3, 9.6)])
def test_5_to_16_tokens_take_the_faster_kernel(gpu, type_, M, N, K, pro, res, tile_us, wide_us):  # noqa: F811
    import torch
    from backpack_amd import capi, kquant
    print("faster kernel", type_, M, N, K, pro, res, flush=True)
    _, _, w = gpu.make_weight(type_, N, K, seed=M)
    X, nw, R = torch.randn(M, K, device="cuda"), torch.rand(K, device="cuda"), torch.randn(M, N, device="cuda")
    if pro or res:
        kquant.matmul_fused(X, w, pro, norm_w=nw if pro else None, eps=1e-5, residual=R if res else None)
    else:
        kquant.matmul(X, w)
    assert (capi.last_form() == "many_token") == (wide_us < tile_us), (capi.last_kernel(), capi.last_form())
