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
    got = kquant.matmul(gpu.dev(X), w, bias=gpu.dev(bias)).cpu().numpy()
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


# pairs per expert around the record sizes (16 .. 64), a skewed routing, one slot per token (whose split X does not fit
# beside the records: the 16-token tile kernel), rows that are no multiple of a workgroup's 256
@pytest.mark.parametrize("tgu,tdn,T,E,k,H,I,skew", [(Q4_K, Q6_K, 5, 8, 2, 256, 256, False), (Q4_K, Q6_K, 17, 2, 2, 512, 256, False),
                                                    (Q5_K, Q5_K, 65, 4, 2, 768, 512, False), (Q6_K, Q4_K, 200, 8, 3, 512, 768, True),
                                                    (Q4_K, Q4_K, 300, 4, 2, 256, 512, False), (Q4_K, Q6_K, 40, 4, 1, 512, 256, False)])
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
    assert capi.last_kernel() == "moe_ffn_mtile"
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


@pytest.mark.parametrize("type_", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("M,N,K", [(1, 1, 256), (17, 255, 512), (33, 257, 2816), (100, 520, 4096), (128, 256, 256), (129, 300, 1024)])
def test_short_prompt_vs_oracle(gpu, kqo, type_, M, N, K):  # noqa: F811
    """bf16 rows of a short prompt: tokens around the groups of 16 and 128, rows around 256, K cut over workgroups and
    not, with a bias; against the oracle on the same bf16 rows and against the GEMM's 128-tile (the same products)."""
    import torch
    from backpack_amd import capi, kquant
    print("short", type_, M, N, K, flush=True)
    raw, packed, w = gpu.make_weight(type_, N, K, seed=M + N)
    rng = np.random.default_rng(K + M)
    X = gpu.dev(rng.standard_normal((M, K)).astype(np.float32)).bfloat16()
    bias = gpu.dev(rng.standard_normal(N).astype(np.float32))
    got = kquant.matmul(X, w, bias=bias).cpu().numpy()
    capi.set_option("gemm_tile", 128)
    try:
        gemm = kquant.matmul(X, w, bias=bias).cpu().numpy()
    finally:
        capi.set_option("gemm_tile", 0)
    want = kqo.matmul(type_, X.float().cpu().numpy(), packed, N, K) + bias.cpu().numpy()
    rms = float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))
    # weights rounded to bf16: 2^-9 per product, K independent ones
    assert np.sqrt(np.mean((got - want) ** 2.0)) <= 2.0 ** -8 * rms
    # the same products in another order: fp32 sums of K of them
    assert np.abs(got - gemm).max() <= 2.0 ** -23 * K ** 0.5 * 8 * max(rms, float(np.abs(want).max()))
