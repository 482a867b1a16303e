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


@pytest.mark.parametrize("M,K,N", [(1, 1, 1), (3, 17, 5), (64, 100, 70), (65, 1, 3), (65, 127, 64),
                                   (66, 128, 65), (70, 129, 1), (130, 1000, 129), (200, 48, 63),
                                   (64, 128, 4097), (1000, 333, 257)])
@pytest.mark.parametrize("form", ["plain", "offset", "strided"])
def test_int_gemm_operands(M, K, N, form):
    """backends.int_gemm on operands of every row length, at odd storage
    offsets and non-contiguous (both transposed views)."""
    from idempotent_llm_amd.backends import int_gemm
    print(f"[int_gemm operands M={M} K={K} N={N} {form}]", flush=True)
    if form == "strided":
        a, b = _i8(M, K + 3, M).t()[:, :K], _i8(N, N, K + 1).t()[:K]
    else:
        off = 3 if form == "offset" else 0
        a = _i8(M, M * K + off + 8)[off:off + M * K].view(M, K)
        b = _i8(N, K * N + off + 8)[off:off + K * N].view(K, N)
    assert torch.equal(int_gemm(a, b, "rocm"), (a.double() @ b.double()).to(torch.int32))


@pytest.mark.parametrize("lead,M,K,N", [((3,), 1, 128, 200), ((2, 4), 33, 128, 65),
                                        ((5,), 64, 60, 31), ((16,), 200, 128, 400), ((0,), 4, 8, 4),
                                        ((2,), 7, 0, 3)])
def test_int_gemm_batched(lead, M, K, N):
    """Batched products, few rows each on the tiled kernel; an empty batch
    and an empty K."""
    from idempotent_llm_amd.backends import int_gemm
    print(f"[int_gemm batched {lead} M={M} K={K} N={N}]", flush=True)
    a = torch.randint(-128, 128, (*lead, M, K), dtype=torch.int8, device="cuda")
    b = torch.randint(-128, 128, (*lead, K, N), dtype=torch.int8, device="cuda")
    want = torch.matmul(a.cpu().double(), b.cpu().double()).to(torch.int32)
    assert torch.equal(int_gemm(a, b, "rocm").cpu(), want)


@pytest.mark.parametrize("K", [130943, 130945, 131056])
def test_int_gemm_longest_k(K):
    """Whole 128-byte slices of these K pass the largest sum (131071) from
    130945 on, where K is padded to 16 only."""
    from idempotent_llm_amd.backends import int_gemm
    print(f"[int_gemm longest K={K}]", flush=True)
    a, b = _i8(1, 65, K), _i8(2, K, 40)
    assert torch.equal(int_gemm(a, b, "rocm"), (a.double() @ b.double()).to(torch.int32))


def test_few_rows_at_any_alignment():
    """detllm_igemm_nt of few rows takes operands at any address."""
    from idempotent_llm_amd._lib import call
    M, N, K = 40, 70, 256
    print("[igemm few rows, operands off by 4 bytes]", flush=True)
    a = _i8(3, M * K + 16)[4:4 + M * K].view(M, K)
    w = _i8(4, N * K + 16)[4:4 + N * K].view(N, K)
    out = torch.empty(M, N, dtype=torch.int32, device="cuda")
    call("detllm_igemm_nt", a, w, out, M, N, K, 1, 0, 0, 0)
    assert torch.equal(out, _want(a, w))


def test_operators_refuse_other_ranks():
    """Operands of another rank raise before any launch."""
    from idempotent_llm_amd import torch_ops  # noqa: F401
    ops = torch.ops.detllm_rocm
    i32, i64, i8 = (torch.zeros(2, 2, 2, 2, 128, dtype=t, device="cuda")
                    for t in (torch.int32, torch.int64, torch.int8))
    v = i64.view(-1)
    for f in (lambda: ops.greedy_pick(i32[0], v), lambda: ops.norm_quant(i32[0], None, 0),
              lambda: ops.swiglu_quant(i32[0], v, v, v, 0, v, 0, v, 0),
              lambda: ops.merge_rowcol(i64[0], v, 0, v, 0),
              lambda: ops.residual_normq(i32[0], v, v, v, 0, 20, i32[0, 0, 0], v, None, 0),
              lambda: ops.attn_prefill(i8, v, i8, i8, i32, i8[0, 0, 0].bool(), 0)):
        with pytest.raises(ValueError):
            f()
    with pytest.raises(ValueError):
        ops.attn_decode(i8[0, 0], v, i8[:, :0], i8, i32[0, 0, 0], i8[0, 0, 0].bool(), 1, i32)


# the lines of the rules that follow K and the alignment of N: four K groups
# from K = 768, 128 x 128 off whole lines of C, 64 x 128 by its tiles, the tile
# columns and N
LINE_CASES = [(512, 1024, 640), (512, 1024, 768), (1501, 4001, 256), (1501, 4001, 1536),
              (1024, 4104, 512), (1024, 4104, 640), (1500, 4016, 128), (3712, 1056, 512),
              (512, 4128, 896), (512, 4128, 1024), (512, 5000, 1024), (1118, 3264, 1152),
              (1408, 1500, 256), (1280, 3113, 256), (1280, 3113, 2048), (900, 3080, 1024),
              (2048, 1271, 1024)]


@pytest.mark.parametrize("M,N,K", LINE_CASES)
def test_tile_rule_lines(M, N, K):
    test_tile_rules(M, N, K)
