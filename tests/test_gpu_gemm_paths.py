"""The int8 products' kernels at the edges of their tile and dispatch rules,
against the product in float64 (sums of int8 products stay below 2^53, so it
is exact). Zero tolerance."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from idempotent_llm_amd import _lib
    _lib.load()


def _i8(seed, *shape):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randint(-128, 128, shape, dtype=torch.int8, device="cuda", generator=g)
    x.view(-1)[:4] = -128
    return x


def _want(a, bt):
    return (a.double() @ bt.double().t()).to(torch.int32)


@pytest.mark.parametrize("M", [1, 16, 17, 33, 49, 64])
@pytest.mark.parametrize("N,K", [(32768, 64), (32775, 1024), (33001, 1040), (32770, 4096)])
def test_head_product(M, N, K):
    """k_gemv_stream at each row-group count, ragged columns, K past one
    1024-byte step and K beyond what its LDS holds at M rows."""
    from idempotent_llm_amd.backends import gemm_nt
    print(f"[head product M={M} N={N} K={K}]", flush=True)
    a, w = _i8(M, M, K), _i8(N + K, N, K)
    out = torch.full((1, M, N), 7, dtype=torch.int32, device="cuda")
    gemm_nt(a, w, out=out)
    assert torch.equal(out[0], _want(a, w))


# (M, N, K) on each side of every tile rule of the prefill product (n = tiles
# of 128 x 64): four K groups, two, none, 128 x 64, 64 x 128, 128 x 128, 128 x
# 192; ragged rows and columns, K of 1, 3, 5 and 9 slices (groups without a
# last slice, groups without any)
TILE_CASES = [(65, 64, 128), (65, 32, 384), (66, 31, 640), (100, 1000, 1152), (512, 1024, 2048),
              (65, 4097, 1024), (129, 2050, 2176), (513, 1024, 3072), (600, 1100, 2304),
              (65, 6144, 1024), (257, 2800, 256), (1025, 1025, 2048), (320, 6144, 384),
              (700, 4099, 1024), (1030, 4096, 640), (1025, 6144, 1024), (2048, 6144, 256)]


@pytest.mark.parametrize("M,N,K", TILE_CASES)
def test_tile_rules(M, N, K):
    from idempotent_llm_amd.backends import gemm_nt
    print(f"[tile rules M={M} N={N} K={K}]", flush=True)
    a, w = _i8(M + K, M, K), _i8(N, N, K)
    out = torch.full((1, M, N), 7, dtype=torch.int32, device="cuda")
    gemm_nt(a, w, out=out)
    assert torch.equal(out[0], _want(a, w))


def test_tile_rules_batched():
    """Batches count as tiles, with batch strides beyond the matrices."""
    from idempotent_llm_amd._lib import call
    print("[tile rules batched]", flush=True)
    for batch, M, N, K in ((3, 70, 100, 640), (16, 512, 200, 128), (5, 130, 1024, 2048)):
        a, w = _i8(batch, batch, M + 1, K), _i8(M, batch, N + 2, K)
        out = torch.full((batch, M + 3, N), 7, dtype=torch.int32, device="cuda")
        call("detllm_igemm_nt", a, w, out, M, N, K, batch, (M + 1) * K, (N + 2) * K, (M + 3) * N)
        for b in range(batch):
            assert torch.equal(out[b, :M], _want(a[b, :M], w[b, :N])), b
        assert (out[:, M:] == 7).all()
