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
                                   (129, 520, 4096)])
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
