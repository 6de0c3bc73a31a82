"""GPU parity of the fp16 / bf16 fused chains against the CPU checker, through the C ABI.

Tolerances (the workload definition's bar): max-abs-err <= 1e-2 and rel-L2 <= 1e-3 against
the fp32/fp64 closed form on identical seeded inputs.  bf16 carries 8 significant bits, so
rounding the softmax probabilities (as the reference does: ``exp(...).astype(in_dtype)``,
bmm_chain.py:63-70) or the output to bf16 alone costs about 1.6e-3 rel-L2; the bf16 cases
therefore assert 1e-3 where no bf16 rounding of P is on the path (cast chains with fp32
output against the checker that rounds the intermediate the same way) and the measured
quantisation figure + 10 % otherwise, always with max-abs-err <= 1e-2.
"""
import numpy as np
import pytest
import torch

from ditto_amd import chain
from tests.gpu_util import errors, report, to_dev, TORCH_DTYPES

pytestmark = pytest.mark.gpu

MAX_ABS = 1e-2
REL_L2 = 1e-3
# bf16 softmax chains (probabilities and output both rounded to bf16): the largest rel-L2 any case of this
# file reaches is 2.36e-3 (1 x 300 x 128 x 128 x 712; the comment above the long-sequence test derives the
# figure from the rounding floor); bound = that + 10 %.  bf16 cast / relu chains meet the stated 1e-3
# against the checker that rounds where they round (measured: at most 1.1e-4).
REL_L2_BF16_QUANT = 2.6e-3
# the same chains with an fp32 output: only the probabilities are rounded to bf16, which costs 1.66e-3 on
# N(0,1) data (tests/test_oracle.py::test_rounding_floor_of_the_16_bit_types); bound = that floor + 5 %, so a
# kernel error of a few 1e-4 cannot hide under the allowance meant for the rounded output
REL_L2_BF16_P_ONLY = 1.75e-3


def bf16_softmax_bound(out_dtype):
    return REL_L2_BF16_P_ONLY if out_dtype == "float32" else REL_L2_BF16_QUANT


def variants(K, N, b_layout="LK"):
    """0 (the library's own choice) and every kernel variant that can run the head size:
    four waves x 32 rows, four waves x 64 rows, eight waves x 32 rows (staggered phases; software
    pipelined; on the 16x16x32 MFMA with 256-row workgroups and with 384-row ones for the first row blocks), four waves with 64-row workgroups on the 16x16x32 MFMA (head
    size up to 64: a wave owns 16 rows and all keys, or 32 rows and half the keys)."""
    pad = 64 if max(K, N) <= 64 else 128
    return [0] + [pad * 10 + q for q in (1, 2, 8, 9, 6, 7) + ((4, 5) if pad == 64 else ())]


def run_chain(A, B, C, dtype, inter, scale=1.0, b_layout="KL", out_dtype=None, variant=0):
    """A[b,M,K], B[b,K,L], C[b,L,N] fp32 numpy (rounded to dtype) -> F numpy fp32."""
    a, c = to_dev(A, dtype), to_dev(C, dtype)
    if b_layout == "LK":  # keep B^T contiguous and hand over the transposed view
        b = to_dev(np.ascontiguousarray(B.transpose(0, 2, 1)), dtype).transpose(1, 2)
    else:
        b = to_dev(B, dtype)
    f = torch.full((A.shape[0], A.shape[1], C.shape[2]), float("nan"), device=a.device,
                   dtype=TORCH_DTYPES[out_dtype or dtype])
    chain.run_bmm_chain(a, b, c, f, inter, scale, tile_variant=variant)
    torch.cuda.synchronize()
    return f.float().cpu().numpy()


SOFTMAX_SHAPES = [
    # batch, M, N, K, L
    (2, 128, 64, 64, 128),
    (3, 200, 64, 64, 136),    # ragged M and L (tail rows / masked keys)
    (2, 96, 40, 72, 200),     # K != N, both padded inside the kernel
    (1, 16, 16, 16, 16),      # smallest shape the reference builders accept
    (2, 512, 64, 64, 512),    # BERT-base head
    (1, 300, 128, 128, 712),  # 128-wide head
    (12, 208, 64, 64, 208),   # ViT-Base/16 row of the reference's shape table
]


@pytest.mark.parametrize("shape", SOFTMAX_SHAPES)
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("b_layout", ["LK", "KL"])
def test_softmax_chain_vs_oracle(oracle, shape, dtype, b_layout):
    batch, M, N, K, L = shape
    scale = 1.0 / np.sqrt(K)
    A, B, C = oracle.make_gemm_chain_inputs(batch, M, N, K, L, dtype, seed=100 + M)
    want = oracle.bmm_chain_f64(A, B, C, inter="softmax", scale=scale)
    for variant in variants(K, N, b_layout):
        for out_dtype in (dtype, "float32"):
            got = run_chain(A, B, C, dtype, "softmax", scale, b_layout, out_dtype, variant)
            assert np.isfinite(got).all(), variant
            mx, rel = errors(got, want)
            if dtype == "bfloat16":
                report("softmax bf16 %s %s variant %d out %s" % (shape, b_layout, variant, out_dtype), mx, rel)
            assert mx <= MAX_ABS, (variant, mx, rel)
            assert rel <= (REL_L2 if dtype == "float16" else bf16_softmax_bound(out_dtype)), (variant, out_dtype, mx, rel)


CAST_SHAPES = [
    (1, 512, 64, 64, 64),     # configuration 1 (shape)
    (2, 128, 64, 64, 128),
    (2, 208, 64, 64, 208),
    (3, 100, 24, 40, 72),     # ragged everything
    (1, 512, 64, 64, 256),    # Mixer-Small row
    (2, 256, 128, 128, 320),
]


@pytest.mark.parametrize("shape", CAST_SHAPES)
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("inter", ["cast", "relu"])
def test_cast_chain_vs_oracle(oracle, shape, dtype, inter):
    batch, M, N, K, L = shape
    A, B, C = oracle.make_gemm_chain_inputs(batch, M, N, K, L, dtype, seed=200 + M, std=0.25)
    # the checker rounds the intermediate to in_dtype exactly where the chain does
    want32 = oracle.bmm_chain_f64(A, B, C, inter=inter, round_mid=dtype)
    want = oracle.np_round_to(want32, dtype)
    for b_layout in ("KL", "LK"):
        for variant in variants(K, N, b_layout):
            got32 = run_chain(A, B, C, dtype, inter, 1.0, b_layout, "float32", variant)
            mx, rel = errors(got32, want32)
            # fp32 accumulation order differs; a rounding flip of one intermediate moves the output
            # by about one unit of the intermediate's last place
            assert mx <= MAX_ABS and rel <= REL_L2, (variant, b_layout, mx, rel)
            got = run_chain(A, B, C, dtype, inter, 1.0, b_layout, None, variant)
            mx, rel = errors(got, want)
            if dtype == "bfloat16":
                report("%s bf16 %s %s variant %d" % (inter, shape, b_layout, variant), mx, rel)
            # one bf16 ulp at |x| ~ 4 is 3e-2
            assert mx <= (MAX_ABS if dtype == "float16" else 4e-2), (variant, b_layout, mx, rel)
            assert rel <= REL_L2, (variant, b_layout, mx, rel)
            # and the narrow output is the rounding of the fp32 output (same kernel, cast at the end)
            assert np.array_equal(got, oracle.np_round_to(got32, dtype)), (variant, b_layout)


@pytest.mark.parametrize("shape", [
    # (batch, M, N, K, L) for the kernel whose waves split the keys: one step of keys and one more key than eight waves take in
    # one, single rows, head sizes at and between its three widths
    (1, 1, 64, 64, 8), (2, 17, 64, 64, 264), (3, 33, 80, 80, 520), (2, 40, 72, 80, 96), (1, 50, 128, 128, 1000),
    (2, 31, 96, 88, 256), (1, 16, 8, 8, 32), (1, 90, 24, 64, 40),
])
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("inter", ["relu", "softmax"])
def test_key_splitting_kernel(oracle, shape, dtype, inter):
    batch, M, N, K, L = shape
    std = 1.0 if inter == "softmax" else 0.25
    A, B, C = oracle.make_gemm_chain_inputs(batch, M, N, K, L, dtype, seed=700 + M + L, std=std)
    # scores that climb past the slack of the running reference within a wave's keys
    B = oracle.np_round_to(B * np.linspace(0.1, 4.0 if inter == "softmax" else 1.0, L, dtype=np.float32)[None, None, :], dtype)
    scale = 0.5 if inter == "softmax" else 1.0
    want = oracle.bmm_chain_f64(A, B, C, inter=inter, scale=scale, round_mid=None if inter == "softmax" else dtype)
    width = 4 if max(K, N) <= 64 else 5 if max(K, N) <= 80 else 8
    for rows in (1, 2):
        variant = 2000 + 10 * width + rows
        for b_layout in ("KL", "LK"):
            got = run_chain(A, B, C, dtype, inter, scale, b_layout, "float32", variant)
            assert np.isfinite(got).all()
            mx, rel = errors(got, want)
            bound = REL_L2 if inter != "softmax" or dtype == "float16" else 2.0e-3  # bf16: the probabilities' own rounding
            assert rel <= bound and mx <= 4e-2, (variant, b_layout, mx, rel)
            narrow = run_chain(A, B, C, dtype, inter, scale, b_layout, dtype, variant)
            assert np.array_equal(narrow, oracle.np_round_to(got, dtype)), (variant, b_layout)


@pytest.mark.parametrize("K", [8, 24, 64, 72, 80, 120, 128])
@pytest.mark.parametrize("b_layout", ["KL", "LK"])
def test_key_splitting_kernel_takes_nothing_from_beside_its_rows(K, b_layout):
    """Rows of A reach the workgroup through LDS, padded to 64, 80 or 128 columns: NaN between and behind the rows stays out, and
    the result is the bits of contiguous rows."""
    gen = torch.Generator(device="cuda").manual_seed(K)
    width = 4 if K <= 64 else 5 if K <= 80 else 8
    for M in (1, 17, 48):
        a, k, v = (torch.randn(2, n, K, device="cuda", generator=gen).half() for n in (M, 40, 40))
        b = k.transpose(1, 2) if b_layout == "LK" else k.transpose(1, 2).contiguous()
        wide = torch.full((2, M + 16, K + 8), float("nan"), device="cuda", dtype=torch.float16)
        view = wide[:, :M, :K]
        view.copy_(a)
        for rows in (1, 2):
            f, g = (torch.full((2, M, K), float("nan"), device="cuda", dtype=torch.float16) for _ in range(2))
            chain.run_bmm_chain(a, b, v, f, "softmax", 0.2, tile_variant=2000 + 10 * width + rows)
            chain.run_bmm_chain(view, b, v, g, "softmax", 0.2, tile_variant=2000 + 10 * width + rows)
            assert torch.isfinite(f).all() and torch.equal(f, g), (M, rows)


@pytest.mark.parametrize("K", [72, 80])
@pytest.mark.parametrize("inter", ["cast", "relu"])
def test_key_splitting_kernel_loads_its_rows_directly(K, inter):
    """16 rows of 65 to 80 columns, B stored [L][K], no softmax: the rows of A take no detour through LDS.  NaN between and behind
    them stays out, the result is the bits of contiguous rows, and the columns' sums are those of 64 bits."""
    gen = torch.Generator(device="cuda").manual_seed(K)
    for M, L in ((1, 31), (16, 32), (17, 257), (70, 300), (300, 600)):
        a, k, v = (torch.randn(2, n, K, device="cuda", generator=gen).half() * 0.25 for n in (M, L, L))
        view = torch.full((2, M + 16, K + 8), float("nan"), device="cuda", dtype=torch.float16)[:, :M, :K]
        view.copy_(a)
        f, g = (torch.full((2, M, K), float("nan"), device="cuda") for _ in range(2))
        chain.run_bmm_chain(a, k.transpose(1, 2), v, f, inter, tile_variant=2051)
        chain.run_bmm_chain(view, k.transpose(1, 2), v, g, inter, tile_variant=2051)
        s = torch.bmm(a.float(), k.float().transpose(1, 2).contiguous()).half().double()
        want = torch.bmm(s.relu() if inter == "relu" else s, v.double())
        # the middle result's rounding alone: 2^-11 of it, and its ties
        assert torch.equal(f, g) and ((f.double() - want).norm() / want.norm()).item() <= 2.0 ** -11, (M, L)


@pytest.mark.parametrize("K,variant", [(8, 2144), (64, 2144), (56, 2148), (72, 2154), (80, 2158), (88, 2188), (128, 2188)])
@pytest.mark.parametrize("b_layout", ["KL", "LK"])
def test_kernel_of_32_rows_a_wave_takes_nothing_from_beside_its_rows(K, variant, b_layout):
    """The same for the kernel of 32 rows a wave: waves of no rows, of one row and of all, one tile of keys and several."""
    gen = torch.Generator(device="cuda").manual_seed(K)
    for M, L in ((1, 40), (33, 64), (300, 200)):
        a, k, v = (torch.randn(2, n, K, device="cuda", generator=gen).half() for n in (M, L, L))
        b = k.transpose(1, 2) if b_layout == "LK" else k.transpose(1, 2).contiguous()
        view = torch.full((2, M + 16, K + 8), float("nan"), device="cuda", dtype=torch.float16)[:, :M, :K]
        view.copy_(a)
        f, g = (torch.full((2, M, K), float("nan"), device="cuda", dtype=torch.float16) for _ in range(2))
        chain.run_bmm_chain(a, b, v, f, "softmax", 0.2, tile_variant=variant)
        chain.run_bmm_chain(view, b, v, g, "softmax", 0.2, tile_variant=variant)
        assert torch.isfinite(f).all() and torch.equal(f, g), (M, L)


@pytest.mark.parametrize("batch,M,L,D,inter,b_layout", [
    # shapes whose kernel is named by its price, on either side of a round of workgroups, ragged rows among them
    (40, 809, 408, 128, "softmax", "LK"), (130, 129, 200, 128, "softmax", "KL"), (5, 432, 144, 128, "relu", "KL"),
    (13, 2049, 200, 128, "cast", "LK"), (65, 416, 416, 64, "relu", "KL"), (160, 300, 296, 64, "cast", "KL"),
    (257, 197, 197, 64, "softmax", "LK"), (3, 49, 176, 64, "cast", "KL"), (2100, 96, 96, 64, "softmax", "LK"),
])
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_kernels_named_by_their_price(oracle, batch, M, L, D, inter, b_layout, dtype):
    std, scale = (1.0, D ** -0.5) if inter == "softmax" else (0.25, 1.0)
    A, B, C = oracle.make_gemm_chain_inputs(batch, M, D, D, L, dtype, seed=M + L, std=std)
    want = oracle.bmm_chain_f64(A, B, C, inter=inter, scale=scale, round_mid=None if inter == "softmax" else dtype)
    got = run_chain(A, B, C, dtype, inter, scale, b_layout, "float32")
    mx, rel = errors(got, want)
    assert np.isfinite(got).all() and mx <= 4e-2, mx
    assert rel <= (REL_L2 if inter != "softmax" or dtype == "float16" else REL_L2_BF16_P_ONLY), rel


@pytest.mark.parametrize("batch,M,L,K,N,inter,b_layout", [
    # few workgroups: the kernel that splits the keys takes them from those of 64 and 128 rows, 16 and 32 rows a workgroup
    (5, 256, 224, 64, 64, "softmax", "KL"), (3, 167, 166, 64, 40, "softmax", "LK"), (1, 513, 96, 56, 64, "cast", "LK"),
    (2, 97, 72, 64, 64, "relu", "KL"), (3, 1553, 272, 128, 128, "softmax", "KL"), (13, 607, 257, 128, 88, "cast", "LK"),
    (3, 1551, 72, 88, 128, "relu", "KL"),
])
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_few_rows_on_the_kernel_that_splits_the_keys(oracle, batch, M, L, K, N, inter, b_layout, dtype):
    std, scale = (1.0, K ** -0.5) if inter == "softmax" else (0.25, 1.0)
    A, B, C = oracle.make_gemm_chain_inputs(batch, M, N, K, L, dtype, seed=M + L, std=std)
    want = oracle.bmm_chain_f64(A, B, C, inter=inter, scale=scale, round_mid=None if inter == "softmax" else dtype)
    bound = REL_L2 if inter != "softmax" or dtype == "float16" else REL_L2_BF16_P_ONLY
    got = run_chain(A, B, C, dtype, inter, scale, b_layout, "float32")
    general = run_chain(A, B, C, dtype, inter, scale, b_layout, "float32", 644 if max(K, N) <= 64 else 1281)
    for result in (got, general):
        mx, rel = errors(result, want)
        assert np.isfinite(result).all() and mx <= 4e-2 and rel <= bound, (mx, rel)
    # the same calls on strided views: row strides above the columns, batches with a gap between
    dt = TORCH_DTYPES[dtype]
    a, c = torch.zeros(batch, M + 3, K + 8, device="cuda", dtype=dt)[:, :M, :K], torch.zeros(batch, L + 1, N + 16, device="cuda", dtype=dt)[:, :L, :N]
    rows = torch.zeros(batch, (K if b_layout == "KL" else L) + 2, (((L + 7) // 8 * 8) if b_layout == "KL" else K) + 8, device="cuda", dtype=dt)
    b = rows[:, :K, :L] if b_layout == "KL" else rows[:, :L, :K].transpose(1, 2)
    for view, values in ((a, A), (b, B), (c, C)):
        view.copy_(to_dev(values, dtype))
    f = torch.full((batch, M + 1, N + 8), float("nan"), device="cuda")[:, :M, :N]
    chain.run_bmm_chain(a, b, c, f, inter, scale)
    assert np.array_equal(f.cpu().numpy(), got)


@pytest.mark.parametrize("batch,M,L,K,N,b_layout,columns", [
    # columns of a workgroup: half, a quarter, a last block of 16, of 8, whole rows where there is nothing to gain or no compute unit left
    (2, 40, 136, 64, 64, "LK", 32), (1, 100, 1112, 64, 64, "KL", 32), (3, 33, 176, 80, 80, "LK", 32), (2, 17, 72, 72, 72, "KL", 32),
    (2, 50, 200, 128, 128, "LK", 32), (5, 200, 264, 128, 128, "LK", 64), (2, 50, 520, 128, 128, "KL", 64), (2, 50, 200, 128, 104, "KL", 32),
    (3, 40, 96, 64, 24, "LK", 24), (9, 300, 64, 64, 64, "LK", 64),
])
@pytest.mark.parametrize("inter", ["softmax", "relu"])
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_key_splitting_kernel_with_columns_shared_out(oracle, batch, M, L, K, N, b_layout, columns, inter, dtype):
    std, scale = (1.0, K ** -0.5) if inter == "softmax" else (0.25, 1.0)
    A, B, C = oracle.make_gemm_chain_inputs(batch, M, N, K, L, dtype, seed=M + L, std=std)
    want = oracle.bmm_chain_f64(A, B, C, inter=inter, scale=scale, round_mid=None if inter == "softmax" else dtype)
    width = 4 if max(K, N) <= 64 else 5 if max(K, N) <= 80 else 8
    t = lambda *s: torch.empty(batch, *s, dtype=TORCH_DTYPES[dtype], device="cuda")
    b = t(K, L) if b_layout == "KL" else t(L, K).transpose(1, 2)
    tile = chain.select_tile(chain.bmm_chain_desc(t(M, K), b, t(L, N), t(M, N), inter, scale, 1.0, 2001 + 10 * width, False))
    assert (tile.variant, tile.block_n) == (2001 + 10 * width, columns)
    got = run_chain(A, B, C, dtype, inter, scale, b_layout, "float32", 2001 + 10 * width)
    mx, rel = errors(got, want)
    assert np.isfinite(got).all() and mx <= 4e-2, mx
    assert rel <= (REL_L2 if inter != "softmax" or dtype == "float16" else REL_L2_BF16_P_ONLY), rel
    narrow = run_chain(A, B, C, dtype, inter, scale, b_layout, dtype, 2001 + 10 * width)
    assert np.array_equal(narrow, oracle.np_round_to(got, dtype))


def masked_scores(oracle, batch, M, N, K, L, dtype, masked, seed):
    """Operands whose scores are minus infinity at the keys ``masked``: column 0 of the first operand is one, and the
    keys hold minus infinity there (how a caller of a chain without a mask argument masks keys)."""
    A, B, C = oracle.make_gemm_chain_inputs(batch, M, N, K, L, dtype, seed=seed)
    A[:, :, 0] = 1.0
    B[:, 0, :] = 0.0
    B[:, 0, masked] = -np.inf
    return A, B, C


# whole groups of a wave's keys without a weight: behind key 100 (padding at the end), the first 96 (padding in front),
# one aligned group alone, all but the last key
MASKED_KEYS = {"end": lambda L: slice(100, L), "front": lambda L: slice(0, 96), "group": lambda L: slice(64, 96),
               "all but one": lambda L: slice(0, L - 1)}

@pytest.mark.parametrize("shape", [(1, 16, 64, 64, 176), (2, 40, 80, 80, 176), (1, 33, 128, 128, 528)])
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("keys", sorted(MASKED_KEYS))
def test_key_splitting_kernel_on_masked_keys(oracle, shape, dtype, keys):
    """A wave whose keys all score minus infinity has no part in the row, whatever the other waves hold (it used to
    make the row NaN: minus infinity less its own reference exponent of minus infinity)."""
    batch, M, N, K, L = shape
    A, B, C = masked_scores(oracle, batch, M, N, K, L, dtype, MASKED_KEYS[keys](L), seed=31 + L)
    want = oracle.bmm_chain_f64(A, B, C, inter="softmax", scale=0.2)
    width = 4 if max(K, N) <= 64 else 5 if max(K, N) <= 80 else 8
    for rows in (1, 2):
        for b_layout in ("KL", "LK"):
            got = run_chain(A, B, C, dtype, "softmax", 0.2, b_layout, "float32", 2000 + 10 * width + rows)
            assert np.isfinite(got).all(), (rows, b_layout)
            mx, rel = errors(got, want)
            # the probabilities' rounding, over as little as one key
            assert mx <= 4e-2 and rel <= (REL_L2 if dtype == "float16" else 2.0e-3), (rows, b_layout, mx, rel)


def test_key_splitting_kernel_masks_rows_one_by_one(oracle):
    """Scores that overflow to minus infinity with the scale, in every other row: those rows' references stay where
    they are while another row of the wave raises its own.  A row without any key is NaN, and only that row."""
    batch, M, N, K, L = 1, 40, 80, 80, 176
    A, B, C = oracle.make_gemm_chain_inputs(batch, M, N, K, L, "bfloat16", seed=5)
    lowest = oracle.np_round_to(np.float32([-3.3e38]), "bfloat16")[0]
    A[:, :, 0] = 0.0
    A[:, ::2, 0] = 1.0
    for masked, none in ((slice(32, L), False), (slice(0, 160), False), (slice(0, L), True)):
        Bm = B.copy()
        Bm[:, 0, :] = 0.0
        Bm[:, 0, masked] = lowest
        want = oracle.bmm_chain_f64(A, Bm, C, inter="softmax", scale=2.0)
        for variant in (2051, 2052):
            got = run_chain(A, Bm, C, "bfloat16", "softmax", 2.0, "LK", "float32", variant)
            rows = slice(1, None, 2) if none else slice(None)
            assert np.isfinite(got[:, rows]).all(), (variant, masked)
            assert not none or np.isnan(got[:, ::2]).all()
            mx, rel = errors(got[:, rows], want[:, rows])
            assert mx <= 4e-2 and rel <= REL_L2_BF16_QUANT, (variant, masked, mx, rel)


@pytest.mark.parametrize("shape", [
    # (batch, M, N, K, L) for the kernel of 32 rows per wave, padded to 64, 80 or 128 columns: a last tile of one half and of two, one tile and more than the
    # ring holds, waves without rows, column counts at and below the padding
    (1, 1, 80, 80, 8), (2, 129, 80, 80, 96), (3, 33, 72, 80, 520), (2, 257, 80, 72, 32), (1, 300, 80, 80, 200), (2, 40, 8, 16, 264),
    (2, 260, 128, 104, 136),  # the 128-column form
])
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("inter", ["relu", "softmax"])
def test_kernel_of_32_rows_per_wave(oracle, shape, dtype, inter):
    batch, M, N, K, L = shape
    std = 1.0 if inter == "softmax" else 0.25
    A, B, C = oracle.make_gemm_chain_inputs(batch, M, N, K, L, dtype, seed=900 + M + L, std=std)
    # scores that climb from key to key: the reference is raised, and with 520 keys the optimistic walk gives way to the exact one
    B = oracle.np_round_to(B * np.linspace(0.1, 6.0 if inter == "softmax" else 1.0, L, dtype=np.float32)[None, None, :], dtype)
    scale = 0.5 if inter == "softmax" else 1.0
    want = oracle.bmm_chain_f64(A, B, C, inter=inter, scale=scale, round_mid=None if inter == "softmax" else dtype)
    for variant in (2144, 2148, 2154, 2158, 2188):
        if variant % 100 // 10 * 16 < max(K, N):
            continue
        for b_layout in ("KL", "LK"):
            got = run_chain(A, B, C, dtype, inter, scale, b_layout, "float32", variant)
            assert np.isfinite(got).all()
            mx, rel = errors(got, want)
            bound = REL_L2 if inter != "softmax" or dtype == "float16" else 2.0e-3  # bf16: the probabilities' own rounding
            assert rel <= bound and mx <= 4e-2, (variant, b_layout, mx, rel)
            narrow = run_chain(A, B, C, dtype, inter, scale, b_layout, dtype, variant)
            assert np.array_equal(narrow, oracle.np_round_to(got, dtype)), (variant, b_layout)


@pytest.mark.parametrize("variant,D", [(2144, 64), (2148, 64), (2154, 80), (2158, 80), (2188, 128)])
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("keys", sorted(MASKED_KEYS))
def test_kernel_of_32_rows_per_wave_on_masked_keys(oracle, variant, D, dtype, keys):
    batch, M, L = 2, 137, 280
    A, B, C = masked_scores(oracle, batch, M, D, D, L, dtype, MASKED_KEYS[keys](L), seed=77 + D)
    want = oracle.bmm_chain_f64(A, B, C, inter="softmax", scale=0.2)
    for b_layout in ("KL", "LK"):
        got = run_chain(A, B, C, dtype, "softmax", 0.2, b_layout, "float32", variant)
        assert np.isfinite(got).all(), b_layout
        mx, rel = errors(got, want)
        assert mx <= 4e-2 and rel <= (REL_L2 if dtype == "float16" else 2.0e-3), (b_layout, mx, rel)


# every kernel that takes several chains a launch, alone and with two levels of batch
@pytest.mark.parametrize("variant,D", [(644, 64), (645, 64), (2041, 64), (2042, 56), (2051, 80), (2052, 72), (2081, 128), (2082, 96),
                                       (2144, 64), (2148, 64), (2154, 80), (2158, 80), (2188, 128)])
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("out", ["own", "float32"])
def test_chains_in_one_launch_on_masked_keys_and_wide_outputs(oracle, variant, D, dtype, out):
    import ctypes

    from ditto_amd import _lib

    batch, M, L, sets, scale = 4, 75, 280, 3, 0.2
    out_dtype = "float32" if out == "float32" else dtype
    dt, lib = TORCH_DTYPES[dtype], _lib.load()
    for keys in sorted(MASKED_KEYS):
        data = [masked_scores(oracle, batch, M, D, D, L, dtype, MASKED_KEYS[keys](L), seed=5 * i + D) for i in range(sets)]
        # A, B as [L][K] and C of a set in one buffer, so that all of them lie equally far from the first set's
        buf = torch.zeros(sets, batch, M + 2 * L, D, device="cuda", dtype=dt)
        for i, (A, B, C) in enumerate(data):
            buf[i] = torch.cat([to_dev(A, dtype), to_dev(np.ascontiguousarray(B.transpose(0, 2, 1)), dtype), to_dev(C, dtype)], 1)
        f = torch.full((sets, batch, M, D), float("nan"), device="cuda", dtype=TORCH_DTYPES[out_dtype])
        for inner in (0, 2):
            x = buf[0].view(2, 2, M + 2 * L, D) if inner else buf[0]
            y = f[0].view(2, 2, M, D) if inner else f[0]
            a, b, c = x[..., :M, :], x[..., M:M + L, :].transpose(-1, -2), x[..., M + L:, :]
            desc = chain.bmm_chain_desc(a, b, c, y, "softmax", scale, 1.0, variant)
            step = buf[0].numel() * buf.element_size()
            at = [[t.data_ptr() + i * step for i in range(sets)] for t in (a, b, c)] + [[f[i].data_ptr() for i in range(sets)]]
            arrays = [(ctypes.c_void_p * sets)(*v) for v in at]
            assert lib.ditto_bmm_chain_sets_launches(ctypes.byref(desc), sets, *arrays) == 1
            f.fill_(float("nan"))
            stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
            assert lib.ditto_bmm_chain_run_sets(ctypes.byref(desc), sets, *arrays, stream) == 0
            torch.cuda.synchronize()
            for i, (A, B, C) in enumerate(data):
                got = f[i].float().cpu().numpy()
                assert np.isfinite(got).all(), (keys, inner, i)
                mx, rel = errors(got, oracle.bmm_chain_f64(A, B, C, inter="softmax", scale=scale))
                # the probabilities' rounding over as little as one key, and the result's own
                assert mx <= 4e-2 and rel <= (REL_L2 if dtype == "float16" else 2.0e-3 if out == "float32" else REL_L2_BF16_QUANT), \
                    (keys, inner, i, mx, rel)


@pytest.mark.parametrize("shape", [(1, 512, 64, 64, 64), (3, 100, 24, 40, 72), (2, 64, 128, 128, 200)])
@pytest.mark.parametrize("inter", ["cast", "relu", "softmax"])
def test_fp32_chain_vs_oracle(oracle, shape, inter):
    # the reference's fp32, CPU-sized configuration (first shape) and ragged ones, fp32 end to end; softmax: the
    # fp32 BMM -> softmax -> BMM of the reference's CPU benchmark (benchmark/chimera/cpu/bmm_softmax_bmm.py:64-170)
    batch, M, N, K, L = shape
    std = 1.0 if inter == "softmax" else 0.25
    A, B, C = oracle.make_gemm_chain_inputs(batch, M, N, K, L, "float32", seed=300 + M, std=std)
    scale = 0.5 if inter == "softmax" else 1.0
    want = oracle.bmm_chain_f64(A, B, C, inter=inter, scale=scale)
    for b_layout in ("KL", "LK"):
        got = run_chain(A, B, C, "float32", inter, scale, b_layout)
        mx, rel = errors(got, want)
        assert mx <= 1e-4 and rel <= 1e-5, (b_layout, mx, rel)  # fp32 sums of <= 200 terms


@pytest.mark.parametrize("shape", [
    # (batch, M, N, K, L): one key, steps of 16 keys that do not fill a round of eight waves, ragged ends of both
    (1, 1, 64, 64, 1), (2, 17, 64, 64, 16), (1, 33, 64, 64, 129), (3, 50, 80, 80, 77), (1, 40, 128, 128, 300),
    (1, 20, 4, 6, 33), (2, 20, 70, 66, 50),   # columns loaded one by one
    (9, 512, 64, 64, 140), (9, 500, 80, 80, 40),  # 32-row workgroups
])
@pytest.mark.parametrize("inter", ["relu", "softmax"])
def test_fp32_chain_at_the_edges_of_its_tiles(oracle, shape, inter):
    batch, M, N, K, L = shape
    A, B, C = oracle.make_gemm_chain_inputs(batch, M, N, K, L, "float32", seed=M + L, std=1.0 if inter == "softmax" else 0.25)
    # scores that climb by far more than the slack of the running reference as the keys go on
    B = B * np.linspace(0.1, 8.0, L, dtype=np.float32)[None, None, :]
    want = oracle.bmm_chain_f64(A, B, C, inter=inter, scale=0.5 if inter == "softmax" else 1.0)
    for b_layout in ("KL", "LK"):
        got = run_chain(A, B, C, "float32", inter, 0.5 if inter == "softmax" else 1.0, b_layout)
        mx, rel = errors(got, want)
        assert np.isfinite(got).all() and rel <= 1e-5, (b_layout, mx, rel)


@pytest.mark.parametrize("shape,width", [
    # (batch, M, N, K, L) and the columns of a workgroup: few rows, more of them, whole rows and ragged ones
    ((1, 33, 64, 64, 40), 16), ((5, 225, 64, 64, 40), 32), ((9, 230, 64, 64, 40), 64), ((5, 225, 50, 60, 40), 32), ((2, 300, 72, 80, 40), 16),
    ((2, 130, 80, 24, 300), 16), ((2, 250, 128, 128, 40), 16), ((3, 250, 128, 128, 40), 32), ((5, 250, 128, 128, 50), 64),
    ((5, 250, 100, 120, 50), 64), ((5, 250, 20, 128, 50), 16),
])
@pytest.mark.parametrize("inter", ["relu", "softmax"])
def test_fp32_chain_with_columns_shared_out(oracle, shape, width, inter):
    batch, M, N, K, L = shape
    d = chain.bmm_chain_desc(*(torch.empty(batch, *s, device="cuda") for s in ((M, K), (K, L), (L, N), (M, N))), inter, 0.5, 1.0, 0, False)
    assert chain.select_tile(d).block_n == width
    test_fp32_chain_at_the_edges_of_its_tiles(oracle, shape, inter)


@pytest.mark.parametrize("shape", [  # (batch, M, columns, L): ends of row tiles and of the waves' steps of 16 keys
    (1, 1, 64, 1), (2, 15, 64, 17), (1, 17, 128, 15), (3, 33, 64, 127), (1, 31, 128, 129), (13, 500, 64, 257), (7, 600, 128, 128)])
@pytest.mark.parametrize("inter", ["cast", "softmax"])
def test_fp32_chain_staged_through_lds(shape, inter):
    """Rows of whole 16-byte pieces reach the fp32 kernel through LDS, others element by element: the same sums, bit for bit."""
    batch, M, D, L = shape
    gen = torch.Generator(device="cuda").manual_seed(M + L)
    q, k, v = (torch.randn(batch, n, D, device="cuda", generator=gen) for n in (M, L, L))
    got = []
    for pad in (0, 4, 1):  # row strides: contiguous, whole pieces, not
        a, b, c = (torch.full((batch, t.shape[1], D + pad), float("nan"), device="cuda")[:, :, :D].copy_(t) for t in (q, k, v))
        f = torch.full((batch, M, D), float("nan"), device="cuda")
        chain.run_bmm_chain(a, b.transpose(1, 2), c, f, inter, 0.2)
        got.append(f)
    assert torch.isfinite(got[0]).all() and torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])


@pytest.mark.parametrize("shape", [  # (batch, M, columns, L): on either side of the keys up to which rows are loaded directly
    (3, 33, 64, 16), (40, 90, 64, 24), (40, 90, 64, 25), (2, 50, 128, 24), (2, 50, 128, 25), (50, 90, 128, 23), (13, 500, 64, 16), (13, 500, 64, 17)])
@pytest.mark.parametrize("inter", ["cast", "relu"])
def test_fp32_chain_of_few_keys(shape, inter):
    test_fp32_chain_staged_through_lds(shape, inter)


@pytest.mark.parametrize("shape", [(44, 429, 64, 111), (52, 469, 64, 51), (45, 621, 56, 65), (31, 813, 80, 130)])  # (batch, M, columns, L)
@pytest.mark.parametrize("inter", ["relu", "softmax"])
def test_fp32_chain_of_two_row_tiles_a_workgroup(shape, inter):
    """B stored [K][L] on 5 rounds of 16-row workgroups against 3 of 32-row ones, and 7 against 4: the 32-row ones run (but for columns
    that are no whole tiles without softmax, up to 64 of them), and give what 64 bits give within the fp32 chain's bound."""
    batch, M, D, L = shape
    gen = torch.Generator(device="cuda").manual_seed(M)
    a, b, c = (torch.randn(batch, *s, device="cuda", generator=gen) for s in ((M, D), (D, L), (L, D)))
    f = torch.full((batch, M, D + 4), float("nan"), device="cuda")[:, :, :D]
    chain.run_bmm_chain(a, b, c, f, inter, 0.2)
    assert chain.select_tile(chain.bmm_chain_desc(a, b, c, f, inter, 0.2)).block_m == (16 if D == 56 and inter == "relu" else 32)
    s = torch.bmm(a.double(), b.double())
    want = torch.bmm(torch.softmax(s * 0.2, -1) if inter == "softmax" else s.relu(), c.double())
    assert torch.isfinite(f).all() and ((f.double() - want).norm() / want.norm()).item() <= 1e-5


@pytest.mark.parametrize("K,N,L,inter,pad,rows", [
    # 7 rounds of 16-row workgroups against 4 of 32: element by element up to 64 columns and beyond, with softmax on either side of 200 keys
    (72, 72, 142, "softmax", 0, 16), (68, 75, 200, "softmax", 0, 16), (72, 72, 201, "softmax", 0, 32), (80, 64, 65, "softmax", 0, 16),
    (64, 80, 33, "cast", 0, 32), (65, 65, 17, "relu", 0, 32), (80, 80, 40, "softmax", 1, 16), (80, 80, 40, "softmax", 4, 32),
    (32, 32, 149, "relu", 0, 16), (63, 64, 31, "softmax", 0, 32), (64, 64, 50, "cast", 1, 16), (64, 64, 50, "cast", 4, 32),
])
def test_fp32_rows_loaded_element_by_element(K, N, L, inter, pad, rows):
    """Two row tiles a workgroup only where they are ahead (`pad`: elements behind the rows of C), within the fp32 chain's bound."""
    gen = torch.Generator(device="cuda").manual_seed(K + L)
    a, b, c = (torch.randn(45, *s, device="cuda", generator=gen) for s in ((619, K), (K, L), (L, N + pad)))
    c[:, :, N:] = float("nan")
    c, f = c[:, :, :N], torch.full((45, 619, N), float("nan"), device="cuda")
    chain.run_bmm_chain(a, b, c, f, inter, 0.2)
    assert chain.select_tile(chain.bmm_chain_desc(a, b, c, f, inter, 0.2)).block_m == rows
    s = torch.bmm(a.double(), b.double())
    want = torch.bmm(torch.softmax(s * 0.2, -1) if inter == "softmax" else s.relu() if inter == "relu" else s, c.double().contiguous())
    assert torch.isfinite(f).all() and ((f.double() - want).norm() / want.norm()).item() <= 1e-5


@pytest.mark.parametrize("shape", [(1, 17, 64, 64, 100), (2, 40, 80, 80, 176), (9, 500, 80, 80, 176), (1, 20, 70, 66, 300), (1, 33, 128, 128, 528)])
@pytest.mark.parametrize("keys", sorted(MASKED_KEYS))
def test_fp32_chain_on_masked_keys(oracle, shape, keys):
    """As above for the fp32 kernel, whose waves take 16 keys at a time."""
    batch, M, N, K, L = shape
    masked = slice(16, L) if keys == "end" and L == 100 else MASKED_KEYS[keys](L)
    A, B, C = masked_scores(oracle, batch, M, N, K, L, "float32", masked, seed=31 + L)
    want = oracle.bmm_chain_f64(A, B, C, inter="softmax", scale=0.2)
    for b_layout in ("KL", "LK"):
        got = run_chain(A, B, C, "float32", "softmax", 0.2, b_layout)
        assert np.isfinite(got).all(), b_layout
        mx, rel = errors(got, want)
        assert rel <= 1e-5, (b_layout, mx, rel)  # fp32 sums, as in the tests above
    # rows without any key are NaN, and only those
    A[:, ::2, 0], A[:, 1::2, 0] = 1.0, 0.0
    B[:, 0, :] = -3.3e38
    got = run_chain(A, B, C, "float32", "softmax", 2.0, "LK")
    assert np.isnan(got[:, ::2]).all() and np.isfinite(got[:, 1::2]).all()


@pytest.mark.parametrize("shape", [(1, 40, 64, 64, 520), (9, 512, 64, 64, 520), (1, 20, 128, 128, 520)])
def test_fp32_chain_on_large_values_and_climbing_scores(oracle, shape):
    """Weights taken relative to a row's maximum are at most one, so a result that fp32 can hold comes out however the
    scores climb: sums of 520 values of 1e34 stay below 1e38."""
    batch, M, N, K, L = shape
    A, B, C = oracle.make_gemm_chain_inputs(batch, M, N, K, L, "float32", seed=M + L)
    B, C = B * np.float32(0.2), C * np.float32(1e34)
    A[:, :, 0] = 1.0
    B[:, 0, :] = 24.0 * (np.arange(L) // 128)  # every wave's next keys score 12 (seventeen binary orders) more
    want = oracle.bmm_chain_f64(A, B, C, inter="softmax", scale=0.5)
    for b_layout in ("KL", "LK"):
        got = run_chain(A, B, C, "float32", "softmax", 0.5, b_layout)
        assert np.isfinite(got).all(), b_layout
        mx, rel = errors(got, want)
        assert rel <= 1e-5, (b_layout, mx, rel)


def test_fp32_chain_beyond_the_work_items_of_one_launch():
    """2^28 rows: 8.4 million workgroups of 512 threads, more than the 2^32 work items a launch holds."""
    M, L, dev = (1 << 28) + 40, 3, "cuda:0"
    gen = torch.Generator(device=dev).manual_seed(8)
    a = torch.randn(1, M, 1, device=dev, generator=gen)
    b, c = (torch.randn(*s, device=dev, generator=gen) for s in ((1, 1, L), (1, L, 1)))
    f = torch.full((1, M, 1), float("nan"), device=dev)
    tile = chain.select_tile(chain.bmm_chain_desc(a, b, c, f, "softmax"))
    assert tile.grid_x * tile.block_threads > 1 << 32
    chain.run_bmm_chain(a, b, c, f, "softmax")
    for at in range(0, M, 1 << 25):
        rows = slice(at, at + (1 << 25))
        want = torch.softmax(a[0, rows] * b[0], -1) @ c[0]
        assert float((f[0, rows] - want).abs().max()) <= 1e-5, at  # fp32 sums of three terms of order one


@pytest.mark.parametrize("shape", [(1, 512, 64, 64, 64), (3, 100, 24, 40, 72), (2, 64, 128, 128, 200)])
@pytest.mark.parametrize("inter", ["cast", "relu", "softmax"])
def test_fp64_chain_vs_oracle(oracle, shape, inter):
    # the reference's ("80", "float64", "float64") row (benchmark/chimera/cuda/bmm_bmm_cuda.py:273-288): doubles end
    # to end, held to the fp64 closed form at 1e-12
    batch, M, N, K, L = shape
    rng = np.random.default_rng(400 + M)
    std = 1.0 if inter == "softmax" else 0.25
    A, B, C = (rng.standard_normal(sh) * std for sh in ((batch, M, K), (batch, K, L), (batch, L, N)))
    scale = 0.5 if inter == "softmax" else 1.0
    mid = A @ B  # (the checker returns single precision: the closed form in numpy doubles here)
    if inter == "relu":
        mid = np.maximum(mid, 0.0)
    elif inter == "softmax":
        e = np.exp(mid * scale - (mid * scale).max(axis=-1, keepdims=True))
        mid = e / e.sum(axis=-1, keepdims=True)
    want = mid @ C
    assert errors(want, oracle.bmm_chain_f64(A, B, C, inter=inter, scale=scale))[1] <= 1e-6
    a, c = torch.from_numpy(A).cuda(), torch.from_numpy(C).cuda()
    for b_layout in ("KL", "LK"):
        b = torch.from_numpy(np.ascontiguousarray(B.transpose(0, 2, 1))).cuda().transpose(1, 2) if b_layout == "LK" \
            else torch.from_numpy(B).cuda()
        f = torch.full((batch, M, N), float("nan"), device="cuda:0", dtype=torch.float64)
        desc = chain.bmm_chain_desc(a, b, c, f, inter, scale)
        assert chain.select_tile(desc).variant == 1001
        chain.run_bmm_chain(a, b, c, f, inter, scale)
        torch.cuda.synchronize()
        got = f.cpu().numpy()
        assert np.abs(got - want).max() <= 1e-12 * max(1.0, np.abs(want).max()), (b_layout, np.abs(got - want).max())
    with pytest.raises(ValueError):  # mixed types are refused
        chain.run_bmm_chain(a, b, c, torch.empty(batch, M, N, device="cuda:0", dtype=torch.float32), inter, scale)


def test_fused_cpu_nest_agrees_with_gpu(oracle):
    # the CPU baseline (the fused loop nest restatement) and the GPU kernel compute the same chain
    A, B, C = oracle.make_gemm_chain_inputs(1, 512, 64, 64, 64, "float16", seed=7, std=0.25)
    cpu = oracle.bmm_chain_fused_f32(A, B, C, inter="cast", round_mid="float16")
    gpu = run_chain(A, B, C, "float16", "cast", out_dtype="float32")
    mx, rel = errors(gpu, cpu)
    assert mx <= MAX_ABS and rel <= REL_L2


@pytest.mark.parametrize("variant", [641, 642, 648, 649, 646, 644, 645])
def test_softmax_invariants_on_gpu(oracle, variant):
    batch, M, N, K, L = 2, 160, 64, 64, 264
    A, B, C = oracle.make_gemm_chain_inputs(batch, M, N, K, L, "float16", seed=9)
    base = run_chain(A, B, C, "float16", "softmax", 0.125, "LK", "float32", variant)
    # V = ones -> O = ones: the normaliser matches the probabilities that were multiplied
    ones = run_chain(A, B, np.ones_like(C), "float16", "softmax", 0.125, "LK", "float32", variant)
    assert np.abs(ones - 1.0).max() <= 2e-3
    # permuting keys and values together leaves O unchanged (up to accumulation order)
    perm = np.random.default_rng(0).permutation(L)
    got = run_chain(A, np.ascontiguousarray(B[:, :, perm]), np.ascontiguousarray(C[:, perm, :]), "float16",
                    "softmax", 0.125, "LK", "float32", variant)
    assert errors(got, base)[1] <= 5e-4
    # Q = 0 -> O = column means of V
    zero = run_chain(np.zeros_like(A), B, C, "float16", "softmax", 0.125, "KL",
                     "float32", variant)
    assert np.abs(zero - C.mean(axis=1, keepdims=True)).max() <= 1e-3
    # large scores do not overflow (the reference's exp-without-max form does)
    Ah = A.copy()
    Ah[:, :, 0] = 60.0
    hot = run_chain(Ah, B, C, "float16", "softmax", 1.0, "LK", "float32", variant)
    want = oracle.bmm_chain_f64(Ah, B, C, inter="softmax", scale=1.0)
    assert np.isfinite(hot).all() and errors(hot, want)[0] <= MAX_ABS


@pytest.mark.parametrize("variant", [0, 641, 642, 648, 649, 646, 647, 644, 645])
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_running_maximum_paths(oracle, variant, dtype):
    """What the lazily raised row maximum has to survive: every score far below zero from the first key on (the
    maximum starts negative), and keys sorted so that every tile of 64 brings a row maximum far above the last
    (a rescale per tile), with ragged M and L.  (The fp16 kernel that pre-scales A keeps scores relative to the
    maximum; the others subtract it per score; the bf16 kernel on the 16x16x32 MFMA takes no maximum per half
    tile but lowers a row's scale when its sum has grown, and repeats the walk with maxima when a sum overflowed.)"""
    batch, M, N, K, L = 2, 200, 64, 64, 456
    rng = np.random.default_rng(5)
    A = rng.standard_normal((batch, M, K)).astype(np.float32)
    B = rng.standard_normal((batch, K, L)).astype(np.float32)
    C = rng.standard_normal((batch, L, N)).astype(np.float32)
    A[:, :, 0] = 4.0
    cases = {}
    Bn = B.copy()
    Bn[:, 0, :] = -24.0                               # q0 k0 = -96: every score around -96 * scale
    cases["all far below zero"] = Bn
    Br = B.copy()
    Br[:, 0, :] = np.linspace(-20.0, 20.0, L)         # the maximum climbs by about 11 per tile at scale 1
    cases["rising"] = Br
    Bf = B.copy()
    Bf[:, 0, :] = np.linspace(20.0, -20.0, L)         # and the other way: later tiles far below the maximum
    cases["falling"] = Bf
    # a jump of 120 in the exponent from one key to the next, and a short spike of 200 inside the first tile:
    # more than an fp32 (or bf16) probability taken relative to the keys before can hold, so a kernel that
    # watches the row sums instead of taking maxima has to notice and walk the keys again the exact way
    Bs = B.copy()
    Bs[:, 0, :] = -15.0
    Bs[:, 0, 300:] = 15.0
    cases["step up"] = Bs
    Bp = B.copy()
    Bp[:, 0, :] = -25.0
    Bp[:, 0, 40:44] = 25.0
    cases["spike in the first tile"] = Bp
    for name, Bx in cases.items():
        Ar, Bxr, Cr = (oracle.np_round_to(t, dtype) for t in (A, Bx, C))
        got = run_chain(Ar, Bxr, Cr, dtype, "softmax", 1.0, "LK", "float32", variant)
        want = oracle.bmm_chain_f64(Ar, Bxr, Cr, inter="softmax", scale=1.0)
        mx, rel = errors(got, want)
        assert np.isfinite(got).all(), name
        assert mx <= MAX_ABS and rel <= (REL_L2_BF16_P_ONLY if dtype == "bfloat16" else REL_L2), (name, mx, rel)


def test_reference_semantics_on_reference_inputs(oracle):
    # the reference's own check: uniform(-1,1) inputs, scale 1, its exp / ones-column / divide
    # form vs torch softmax at rtol = atol = 0.1 (testing/hyper_fusion/bmm_softmax_bmm_wmma_...py:552-587)
    rng = np.random.default_rng(3)
    batch, M, N, K, L = 12, 512, 64, 64, 512
    A = oracle.np_round_to(rng.uniform(-1, 1, (batch, M, K)).astype(np.float32), "float16")
    B = oracle.np_round_to(rng.uniform(-1, 1, (batch, K, L)).astype(np.float32), "float16")
    C = oracle.np_round_to(rng.uniform(-1, 1, (batch, L, N)).astype(np.float32), "float16")
    emul = oracle.bmm_softmax_ref_emul(A, B, C, "float16")
    got = run_chain(A, B, C, "float16", "softmax", 1.0, "KL")
    assert np.isfinite(got).all()
    # the reference's form breaks where exp or its row sum exceeds the fp16 range (65504): a
    # score above 11.09 gives inf/nan ("nan errors occurs", same file :612-613), a row sum above
    # 65504 an infinite divisor.  Compare on the rows where its form is representable.
    den = np.exp(A.astype(np.float64) @ B.astype(np.float64)).sum(axis=-1)
    ok = np.isfinite(emul).all(axis=-1) & (den < 60000.0)
    assert 0.95 < ok.mean() < 1.0
    assert np.allclose(got[ok], emul[ok], rtol=0.1, atol=0.1)
    assert errors(got[ok], emul[ok])[0] <= 5e-3


def test_attention_full_size_fp16_heads(oracle):
    # the fp16 configuration at its full size: 96 heads of 512 x 64, scale 1/8, every row checked
    batch, M, N, K, L = 96, 512, 64, 64, 512
    A, B, C = oracle.make_gemm_chain_inputs(batch, M, N, K, L, "float16", seed=21)
    want = oracle.bmm_chain_f64(A, B, C, inter="softmax", scale=0.125)
    for variant in variants(K, N):
        got = run_chain(A, B, C, "float16", "softmax", 0.125, "LK", None, variant)
        mx, rel = errors(got, want)
        report("attention fp16 96 x 512 x 64, variant %d" % variant, mx, rel)
        assert mx <= MAX_ABS and rel <= REL_L2, (variant, mx, rel)


# Measured on the long-sequence configuration (64 heads of 4096 x 128, N(0,1) inputs, scale 1/sqrt(128)),
# the same for the three kernel variants to two digits: bf16 rel-L2 2.33e-3 .. 2.35e-3 (max-abs 3.9e-4 ..
# 4.9e-4), fp16 rel-L2 2.87e-4 .. 2.95e-4 (max-abs 4.7e-5 .. 7.0e-5).  The rel-L2 bounds are the largest
# measured figure + 10 %; max-abs, a maximum over a million outputs, gets twice the largest figure.
# The bf16 figure is rounding, not the online softmax: rounding N(0,1) data to bf16 costs rel-L2 1.66e-3 by
# itself (tests/test_oracle.py::test_rounding_floor_of_the_16_bit_types), the chain rounds both the
# probabilities and the output, and 1.66e-3 * sqrt(2) = 2.35e-3.  The fp16 run of the same shape holds the
# online softmax itself, 64 steps and their rescales per row, to the stated 1e-3.
MAX_ABS_BF16_LONG, REL_L2_BF16_LONG = 1.0e-3, 2.6e-3
MAX_ABS_FP16_LONG, REL_L2_FP16_LONG = 1.4e-4, 3.25e-4


@pytest.mark.parametrize("variant", [0, 1282, 1288, 1289, 1286, 1287])
def test_attention_full_size_fp16_long_sequence(oracle, variant):
    # the long-sequence shape in fp16, where the stated bar (1e-2 / 1e-3) is reachable: 64 online-softmax
    # steps per row, every variant; three whole heads and a row block of every head against the closed form
    batch, S, d = 64, 4096, 128
    scale = d ** -0.5
    dev = "cuda:0"
    g = torch.Generator(device="cpu").manual_seed(34)
    q = torch.randn(batch, S, d, generator=g).to(torch.float16)
    k = torch.randn(batch, S, d, generator=g).to(torch.float16)
    v = torch.randn(batch, S, d, generator=g).to(torch.float16)
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    out = torch.full((batch, S, d), float("nan"), device=dev, dtype=torch.float16)
    chain.run_bmm_chain(qd, kd.transpose(1, 2), vd, out, "softmax", scale, tile_variant=variant)
    torch.cuda.synchronize()
    got = out.float().cpu().numpy()
    assert np.isfinite(got).all()
    qn, kn, vn = q.float().numpy(), k.float().numpy(), v.float().numpy()
    for h in (0, 17, 63):
        want = oracle.bmm_chain_f64(qn[h:h + 1], np.ascontiguousarray(kn[h:h + 1].transpose(0, 2, 1)), vn[h:h + 1],
                                    inter="softmax", scale=scale)
        mx, rel = errors(got[h:h + 1], want)
        report("attention fp16 64 x 4096 x 128, variant %d, head %d" % (variant, h), mx, rel)
        assert mx <= MAX_ABS and rel <= REL_L2, (h, mx, rel)                      # the stated bar
        assert mx <= MAX_ABS_FP16_LONG and rel <= REL_L2_FP16_LONG, (h, mx, rel)  # measured + 10 %
    rows = slice(3000, 3032)
    want = oracle.bmm_chain_f64(np.ascontiguousarray(qn[:, rows]), np.ascontiguousarray(kn.transpose(0, 2, 1)), vn,
                                inter="softmax", scale=scale)
    mx, rel = errors(got[:, rows], want)
    report("attention fp16 64 x 4096 x 128, variant %d, rows 3000-3031 of every head" % variant, mx, rel)
    assert mx <= MAX_ABS_FP16_LONG and rel <= REL_L2_FP16_LONG, (mx, rel)
    # scores shifted far from zero: keys scaled up make row maxima of +-40 and more in the exponent, so
    # the running maximum is raised many times along a row
    big = (kd.float() * 6.0).to(torch.float16)
    chain.run_bmm_chain(qd[:2], big[:2].transpose(1, 2), vd[:2], out[:2], "softmax", scale, tile_variant=variant)
    torch.cuda.synchronize()
    want = oracle.bmm_chain_f64(qn[:2, :256], np.ascontiguousarray(big[:2].float().cpu().numpy().transpose(0, 2, 1)),
                                vn[:2], inter="softmax", scale=scale)
    mx, rel = errors(out[:2, :256].float().cpu().numpy(), want)
    report("attention fp16 2 x 4096 x 128 with keys x 6, variant %d" % variant, mx, rel)
    assert mx <= MAX_ABS and rel <= REL_L2, (mx, rel)


@pytest.mark.parametrize("variant", [0, 1282, 1288, 1289, 1286, 1287])
def test_attention_full_size_bf16_long_sequence(oracle, variant):
    # the bf16 configuration at its full size (64 heads of 4096 x 128).  The CPU closed form over
    # all of it would take minutes, so: every row of three heads chosen across the batch, one
    # row block of every head, and size-independent properties over the whole output.
    batch, S, d = 64, 4096, 128
    scale = d ** -0.5
    dev = "cuda:0"
    g = torch.Generator(device="cpu").manual_seed(33)
    q = torch.randn(batch, S, d, generator=g).to(torch.bfloat16)
    k = torch.randn(batch, S, d, generator=g).to(torch.bfloat16)
    v = torch.randn(batch, S, d, generator=g).to(torch.bfloat16)
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    out = torch.full((batch, S, d), float("nan"), device=dev, dtype=torch.bfloat16)
    chain.run_bmm_chain(qd, kd.transpose(1, 2), vd, out, "softmax", scale, tile_variant=variant)
    torch.cuda.synchronize()
    got = out.float().cpu().numpy()
    assert np.isfinite(got).all()
    qn, kn, vn = q.float().numpy(), k.float().numpy(), v.float().numpy()
    for h in (0, 31, 63):  # whole heads
        want = oracle.bmm_chain_f64(qn[h:h + 1], np.ascontiguousarray(kn[h:h + 1].transpose(0, 2, 1)), vn[h:h + 1],
                                    inter="softmax", scale=scale)
        mx, rel = errors(got[h:h + 1], want)
        report("attention bf16 64 x 4096 x 128, variant %d, head %d" % (variant, h), mx, rel)
        assert mx <= MAX_ABS_BF16_LONG and rel <= REL_L2_BF16_LONG, (h, mx, rel)
    rows = slice(1000, 1032)  # one row block of every head (straddles no tile boundary specially)
    want = oracle.bmm_chain_f64(np.ascontiguousarray(qn[:, rows]), np.ascontiguousarray(kn.transpose(0, 2, 1)), vn,
                                inter="softmax", scale=scale)
    mx, rel = errors(got[:, rows], want)
    report("attention bf16 64 x 4096 x 128, variant %d, rows 1000-1031 of every head" % variant, mx, rel)
    assert mx <= MAX_ABS_BF16_LONG and rel <= REL_L2_BF16_LONG, (mx, rel)
    # values all ones -> output all ones (the normaliser is the sum of what was multiplied)
    ones = torch.ones_like(vd)
    chain.run_bmm_chain(qd, kd.transpose(1, 2), ones, out, "softmax", scale, tile_variant=variant)
    torch.cuda.synchronize()
    assert (out.float() - 1.0).abs().max().item() <= 8e-3  # one bf16 ulp below 1 is 3.9e-3
    # convexity: every output lies within the column range of V of its head
    chain.run_bmm_chain(qd, kd.transpose(1, 2), vd, out, "softmax", scale, tile_variant=variant)
    torch.cuda.synchronize()
    lo = vd.float().amin(dim=1, keepdim=True)
    hi = vd.float().amax(dim=1, keepdim=True)
    o32 = out.float()
    assert bool(((o32 >= lo - 1e-2) & (o32 <= hi + 1e-2)).all())
    # rows of Q permuted -> rows of the output permuted the same way.  Not bit for bit: the
    # running maximum is raised for all rows of a wave at once, so a row's rescale history (and
    # with it the last bit before rounding) depends on its neighbours; a few outputs move by
    # one bf16 unit in the last place.
    perm = torch.randperm(S, generator=g).to(dev)
    out2 = torch.empty_like(out)
    chain.run_bmm_chain(qd[:, perm].contiguous(), kd.transpose(1, 2), vd, out2, "softmax", scale, tile_variant=variant)
    torch.cuda.synchronize()
    a, b = out2.float(), out[:, perm].float()
    assert float((a != b).float().mean()) <= 1e-2
    assert float((a - b).norm() / b.norm()) <= 5e-4
    assert bool(((a - b).abs() <= 2.0 ** -7 * b.abs() + 1e-6).all())


@pytest.mark.parametrize("variant", [0, 1281, 1288, 1289])
def test_gemm_chain_full_size_bf16(oracle, variant):
    # the large GEMM-chain point of the benchmark, (A.B).D with the cast between, 64 x (4096 x 128 x
    # 4096 x 128) bf16, B as [K][L] like the reference's operand.  The checker over all of it would take
    # minutes: whole entries across the batch, one row block of every entry, and properties.
    batch, M, K, L, N = 64, 4096, 128, 4096, 128
    dev = "cuda:0"
    g = torch.Generator(device="cpu").manual_seed(35)
    a = (torch.randn(batch, M, K, generator=g) * 0.25).to(torch.bfloat16)
    b = (torch.randn(batch, K, L, generator=g) * 0.25).to(torch.bfloat16)
    c = (torch.randn(batch, L, N, generator=g) / 64).to(torch.bfloat16)  # keeps the outputs O(1)
    ad, bd, cd = a.to(dev), b.to(dev), c.to(dev)
    out = torch.full((batch, M, N), float("nan"), device=dev, dtype=torch.bfloat16)
    chain.run_bmm_chain(ad, bd, cd, out, "cast", 1.0, tile_variant=variant)
    torch.cuda.synchronize()
    got = out.float().cpu().numpy()
    assert np.isfinite(got).all()
    an, bn, cn = a.float().numpy(), b.float().numpy(), c.float().numpy()
    for h in (0, 40, 63):
        want = oracle.bmm_chain_f64(an[h:h + 1], bn[h:h + 1], cn[h:h + 1], inter="cast", round_mid="bfloat16")
        mx, rel = errors(got[h:h + 1], oracle.np_round_to(want.astype(np.float32), "bfloat16"))
        report("GEMM chain bf16 64 x 4096 x 128, variant %d, head %d" % (variant, h), mx, rel)
        assert rel <= REL_L2 and mx <= 4e-2, (h, mx, rel)  # one bf16 ulp at |x| ~ 4 is 3e-2
    rows = slice(3000, 3040)
    want = oracle.bmm_chain_f64(np.ascontiguousarray(an[:, rows]), bn, cn, inter="cast", round_mid="bfloat16")
    mx, rel = errors(got[:, rows], oracle.np_round_to(want.astype(np.float32), "bfloat16"))
    assert rel <= REL_L2 and mx <= 4e-2, (mx, rel)
    # B = [I | 0]: the middle result is A itself (exact in bf16), so F = A . C[:K] -- one GEMM
    eye = torch.zeros(batch, K, L, dtype=torch.bfloat16, device=dev)
    eye[:, torch.arange(K), torch.arange(K)] = 1
    chain.run_bmm_chain(ad, eye, cd, out, "cast", 1.0, tile_variant=variant)
    torch.cuda.synchronize()
    want_d = torch.bmm(ad.float(), cd[:, :K].float())
    # (against an unrounded fp32 product: the bf16 rounding of the output alone is 1.66e-3)
    assert float((out.float() - want_d).norm() / want_d.norm()) <= REL_L2_BF16_QUANT
    # rows of A permuted -> rows of F permuted, bit for bit (no cross-row state in this chain)
    perm = torch.randperm(M, generator=g).to(dev)
    chain.run_bmm_chain(ad, bd, cd, out, "cast", 1.0, tile_variant=variant)
    out2 = torch.empty_like(out)
    chain.run_bmm_chain(ad[:, perm].contiguous(), bd, cd, out2, "cast", 1.0, tile_variant=variant)
    torch.cuda.synchronize()
    assert torch.equal(out2, out[:, perm])


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("cfg", [(2, 3, 200, 64), (1, 16, 256, 128), (8, 12, 512, 64)])
def test_multi_head_attention_module(oracle, dtype, cfg):
    # packed [batch, M, 3*hidden] projection in, [batch, M, hidden] out, heads walked by stride;
    # checked against the reference's own formulation (split, reshape, transpose, chain, merge:
    # nn/module/self_attention.py:46-73) evaluated in fp64 on the CPU
    from ditto_amd import auto_compute as ac

    batch, heads, M, d = cfg
    hidden = heads * d
    rng = np.random.default_rng(heads + M)
    qkv = oracle.np_round_to(rng.standard_normal((batch, M, 3 * hidden)).astype(np.float32), dtype)
    mha = ac.nn.module.MultiHeadAttentionMMA(heads, hidden, in_dtype=dtype, scale=None)
    x = to_dev(qkv, dtype)
    out = mha(x)
    torch.cuda.synchronize()
    assert out.shape == (batch, M, hidden) and out.is_contiguous()
    q, k, v = (qkv[:, :, i * hidden:(i + 1) * hidden].reshape(batch, M, heads, d).transpose(0, 2, 1, 3)
               .reshape(batch * heads, M, d) for i in range(3))
    want = oracle.bmm_chain_f64(q, np.ascontiguousarray(k.transpose(0, 2, 1)), v, inter="softmax", scale=d ** -0.5)
    want = want.reshape(batch, heads, M, d).transpose(0, 2, 1, 3).reshape(batch, M, hidden)
    mx, rel = errors(out.float().cpu().numpy(), want)
    if dtype == "bfloat16":
        report("multi-head attention bf16 %s" % (cfg,), mx, rel)
    assert mx <= MAX_ABS and rel <= (REL_L2 if dtype == "float16" else REL_L2_BF16_QUANT), (mx, rel)
    # same numbers as the chain on materialised per-head tensors (bit for bit: same kernel, same order)
    qd, kd, vd = (to_dev(np.ascontiguousarray(t), dtype) for t in (q, k, v))
    ref = torch.empty(batch * heads, M, d, device=x.device, dtype=x.dtype)
    chain.run_bmm_chain(qd, kd.transpose(1, 2), vd, ref, "softmax", d ** -0.5,
                        tile_variant=chain.select_tile(chain.bmm_chain_desc(*mha.head_views(x), out.view(batch, M, heads, d).permute(0, 2, 1, 3), "softmax", d ** -0.5)).variant)
    torch.cuda.synchronize()
    assert torch.equal(ref.view(batch, heads, M, d).permute(0, 2, 1, 3).reshape(batch, M, hidden), out)


def test_tile_variant_tuning_round_trip(tmp_path, oracle):
    # measure the variants for one shape, log them in the reference's format, reuse the log
    from ditto_amd.auto_schedule.schedulers import chimera_integrate as ci

    dev = "cuda:0"
    torch.manual_seed(1)
    q, k, v = (torch.randn(16, 1024, 64, device=dev).half() for _ in range(3))
    f = torch.empty_like(q)
    log = str(tmp_path / "chimera_tune.log")
    key = ci.workload_key(chain.bmm_chain_desc(q, k.transpose(1, 2), v, f, "softmax", 0.125))
    best = ci.select_tile_variant(key, log, q, k.transpose(1, 2), v, f, "softmax", 0.125, top=3, min_repeat_ms=5)
    records = ci.load_best_records(log)
    assert len(open(log).read().strip().splitlines()) == 3
    assert records[key]["record"]["variant"] == best.record["variant"] and 0 < best.value < 5.0
    assert ci.auto_schedule_bmm_chain_hip(key, log, q, k.transpose(1, 2), v, f, "softmax", 0.125) == best.record["variant"]
    chain.run_bmm_chain(q, k.transpose(1, 2), v, f, "softmax", 0.125, tile_variant=best.record["variant"])
    ref = torch.softmax(q.float() @ k.float().transpose(1, 2) * 0.125, -1) @ v.float()
    assert (f.float() - ref).abs().max().item() <= MAX_ABS


def test_tuning_heads_of_80_columns(tmp_path, oracle):
    # ViT-Huge attention: the kernels padded to 80 columns are measured, the library's own among them
    from ditto_amd.auto_schedule.schedulers import chimera_integrate as ci

    A, B, C = oracle.make_gemm_chain_inputs(16, 197, 80, 80, 197, "float16", seed=2)
    q, k, v = to_dev(A, "float16"), to_dev(np.ascontiguousarray(B.transpose(0, 2, 1)), "float16"), to_dev(C, "float16")
    f = torch.empty_like(q)
    log = str(tmp_path / "chimera_80.log")
    desc = chain.bmm_chain_desc(q, k.transpose(1, 2), v, f, "softmax", 80 ** -0.5)
    key = ci.workload_key(desc)
    variant = ci.auto_schedule_bmm_chain_hip(key, log, q, k.transpose(1, 2), v, f, "softmax", 80 ** -0.5)
    # (fp32 has one kernel: tuning measures it)
    q32, k32, v32, f32 = (t.float() for t in (q, k, v, f))
    assert ci.auto_schedule_bmm_chain_hip("fp32", str(tmp_path / "f32.log"), q32, k32.transpose(1, 2), v32, f32) == 1000
    lines = open(log).read().strip().splitlines()
    assert len(lines) == 3 and '"variant": %d' % chain.select_tile(desc).variant in lines[0]
    f.fill_(float("nan"))
    chain.run_bmm_chain(q, k.transpose(1, 2), v, f, "softmax", 80 ** -0.5, tile_variant=variant)
    want = oracle.bmm_chain_f64(A, B, C, inter="softmax", scale=80 ** -0.5)
    assert errors(f.float().cpu().numpy(), want)[1] <= REL_L2


def test_strided_views_and_errors():
    dev = "cuda:0"
    torch.manual_seed(0)
    # operands that are slices of larger buffers (row stride > row extent)
    big_a = torch.randn(2, 128, 96, device=dev).half()
    big_b = torch.randn(2, 160, 96, device=dev).half()
    big_c = torch.randn(2, 160, 96, device=dev).half()
    a, bt, c = big_a[:, :, :64], big_b[:, :, 16:80], big_c[:, :, 8:72]
    f = torch.empty(2, 128, 64, device=dev, dtype=torch.float16)
    chain.run_bmm_chain(a, bt.transpose(1, 2), c, f, "softmax", 0.125)
    ref = torch.softmax(a.float() @ bt.float().transpose(1, 2) * 0.125, -1) @ c.float()
    assert (f.float() - ref).abs().max().item() <= MAX_ABS
    # the output as a slice too.  Rows that all start on 16 bytes (row stride 96) leave through LDS as whole rows,
    # others (row stride 100) are stored from registers, four columns per lane: every variant gives the same bits
    for variant in variants(64, 64, "LK"):
        chain.run_bmm_chain(a, bt.transpose(1, 2), c, f, "softmax", 0.125, tile_variant=variant)
        for width in (96, 100):
            big_f = torch.full((2, 128, width), float("nan"), device=dev, dtype=torch.float16)
            chain.run_bmm_chain(a, bt.transpose(1, 2), c, big_f[:, :, 8:72], "softmax", 0.125, tile_variant=variant)
            assert torch.equal(big_f[:, :, 8:72], f), (variant, width)
            assert torch.isnan(big_f[:, :, :8]).all() and torch.isnan(big_f[:, :, 72:]).all(), (variant, width)
    with pytest.raises(ValueError):
        chain.run_bmm_chain(a[:, :, :60], bt[:, :, :60].transpose(1, 2), c, f, "softmax", 0.125)
    with pytest.raises(ValueError):
        chain.run_bmm_chain(a, bt.transpose(1, 2), c, f[:, :64], "softmax", 0.125)
    with pytest.raises(NotImplementedError):
        wide = torch.randn(2, 128, 256, device=dev).half()
        chain.run_bmm_chain(wide, torch.randn(2, 256, 64, device=dev).half(),
                            torch.randn(2, 64, 64, device=dev).half(), f, "cast")
    with pytest.raises(ValueError):
        chain.run_bmm_chain(a.cpu(), bt.transpose(1, 2).cpu(), c.cpu(), f.cpu(), "softmax", 0.125)


def test_fp16_accumulator_request_is_served_in_fp32():
    """The reference's ("80", "float16", "float16") rows (benchmark/chimera/cuda/bmm_bmm_cuda.py:273-288): an fp16
    accumulator asked for with fp16 operands runs the same kernels on the MFMA's fp32 accumulator -- the same bits as
    the fp32 request; a bf16 accumulator is no row of the reference and stays refused."""
    from ditto_amd import _lib
    dev = "cuda:0"
    torch.manual_seed(1)
    a, bt, c = (torch.randn(2, 128, 64, device=dev).half() for _ in range(3))
    f32, f16 = (torch.empty(2, 128, 64, device=dev, dtype=torch.float16) for _ in range(2))
    for inter in ("softmax", "cast"):
        chain.run_bmm_chain(a, bt.transpose(1, 2), c, f32, inter, 0.125)
        desc = chain.bmm_chain_desc(a, bt.transpose(1, 2), c, f16, inter, 0.125)
        desc.acc_dtype = _lib.F16
        chain.run_bmm_chain(a, bt.transpose(1, 2), c, f16, inter, 0.125, desc=desc)
        assert torch.equal(f16, f32)
    ab, bb, cb = a.bfloat16(), bt.bfloat16(), c.bfloat16()
    fb = torch.empty(2, 128, 64, device=dev, dtype=torch.bfloat16)
    desc = chain.bmm_chain_desc(ab, bb.transpose(1, 2), cb, fb, "cast")
    desc.acc_dtype = _lib.BF16
    with pytest.raises(NotImplementedError):
        chain.run_bmm_chain(ab, bb.transpose(1, 2), cb, fb, "cast", desc=desc)


def test_front_end_end_to_end(oracle):
    import ditto_amd as ditto
    from ditto_amd import auto_compute as ac, auto_tensorize as at, hardware as hw

    batch, M, N, K, L = 8, 256, 64, 64, 256
    ins, outs = ac.nn.functional.BatchGemmSoftmaxGemm(batch, M, N, K, L, "float16", "float32", scale=0.125)
    A, B, C = ins
    (F,) = outs
    E_frag = F.op.input_tensors[0]
    exp, C_ext = E_frag.op.input_tensors
    D_frag = exp.op.input_tensors[0]
    b, m, n, mi, ni = E_frag.op.axis
    rlo, rli = E_frag.op.reduce_axis
    fuse_choice = at.fusion_choice(D_frag.op, E_frag.op, [b, m, n, rlo, mi, ni, rli], 3)
    p1 = at.cuda_wmma(16, 16, 16, "float16", "float32", "shared")
    p2 = at.cuda_wmma(16, 16, 16, "float16", "float32", "global")
    layer = ac.layer([F.op], inputs=[A, B, C])
    state = at.tensorize_hyper_fusion_state(layer, fuse_choice, {
        D_frag.op: at.match_info(at.intrinsic_match(D_frag, p1, ["InnerMost", "SameRange"])[0], p1),
        E_frag.op: at.match_info(at.intrinsic_match(E_frag, p2, ["InnerMost", "SameRange"])[0], p2)})
    sch = at.tensorize_cuda(layer, state, hw.query_hw_param("gpu.hip.MI355X"), at.cuda_tensorize_param())
    func = ditto.build(sch, layer.schedule_tensors, "hip")
    a_np, b_np, c_np = oracle.make_gemm_chain_inputs(batch, M, N, K, L, "float16", seed=5)
    args = [to_dev(a_np, "float16"), to_dev(b_np, "float16"), to_dev(c_np, "float16"),
            torch.empty(batch, M, N, device="cuda:0", dtype=torch.float16)]
    func(*args)
    torch.cuda.synchronize()
    want = oracle.bmm_chain_f64(a_np, b_np, c_np, inter="softmax", scale=0.125)
    mx, rel = errors(args[3].float().cpu().numpy(), want)
    assert mx <= MAX_ABS and rel <= REL_L2
    t = func.time_evaluator(func.entry_name, None, min_repeat_ms=20)(*args)
    assert 0 < t.mean < 1e-2
    with pytest.raises(ValueError):
        func(*args[:3])


def test_reference_test_flow_with_build_fusion_choice(oracle):
    """python_test/auto_tensorize/test_hyper_fusion.py:833-910 (test_tensorize_cuda_run) against this package:
    serial fusion state -> intrinsic match -> register_tensorize_axes -> build_fusion_choice ->
    tensorize_hyper_fusion_state -> tensorize_cuda -> build -> time_evaluator, on the reference's own
    uniform(-1, 1) inputs; the result is checked, which the reference's test does not do."""
    import ditto_amd as ditto
    from ditto_amd import auto_compute as ac, auto_tensorize as at, hardware as hw

    ins, outs = ac.nn.functional.BatchGemmSoftmaxGemm()  # the reference's defaults: 12 x 512 x 64 x 64 x 512
    layer = ac.layer([outs[0].op], inputs=ins)
    sfs = at.build_serial_fusion_state(layer)
    op1, op2 = sfs.first_op, sfs.second_op

    def get_match_info(op, store_scope):
        packed = at.cuda_wmma(16, 16, 16, "float16", "float32", store_scope)
        choice = at.intrinsic_match(op.output(0), packed, ["InnerMost", "SameRange"])[0]
        return at.match_info(choice, packed, impl="")

    first_match_info = get_match_info(op1, "shared")
    second_match_info = get_match_info(op2, "global")
    sfs.register_tensorize_axes(list(first_match_info.axis) + list(second_match_info.axis))
    V100 = hw.query_hw_param("gpu.cuda.V100")
    fuse_choice = at.build_fusion_choice(sfs, hw_param=V100, dtype="float32", simple_mode=-1)
    tensorize_state = at.tensorize_hyper_fusion_state(layer, fuse_choice, {op1: first_match_info, op2: second_match_info})
    tensorize_param = at.cuda_tensorize_param(warp_size=32, ty_size=4, tz_size=2, input_vector_len=4, serial_y=2,
                                              serial_z=1, block_rx=8, warp_rx=4, block_ry=1, warp_ry=4,
                                              unroll_steps=512)
    sch = at.tensorize_cuda(layer, tensorize_state, V100, tensorize_param)
    func = ditto.build(sch, layer.schedule_tensors, "hip")
    rng = np.random.default_rng(0)
    inputs_np = [oracle.np_round_to(rng.uniform(-1, 1, [int(x) for x in y.shape]).astype(np.float32), "float16")
                 for y in ins]
    inputs = [to_dev(x, "float16") for x in inputs_np]
    outputs = [torch.full(tuple(y.shape), float("nan"), device="cuda:0", dtype=torch.float16) for y in outs]
    evaluator = func.time_evaluator(func.entry_name, None, min_repeat_ms=50)
    cost = evaluator(*inputs, *outputs).mean * 1e3
    assert 0 < cost < 1.0  # ms
    want = oracle.bmm_chain_f64(*inputs_np, inter="softmax", scale=1.0)
    mx, rel = errors(outputs[0].float().cpu().numpy(), want)
    assert mx <= MAX_ABS and rel <= REL_L2, (mx, rel)
    # the descriptor is filled once and reused; a forced variant travels from the schedule to the call
    assert len(func._descs) == 1
    sch8 = at.tensorize_hip(layer, tensorize_state, tile_variant=648)
    f8 = ditto.build(sch8, layer.schedule_tensors, "hip")
    f8(*inputs, *outputs)
    torch.cuda.synchronize()
    assert next(iter(f8._descs.values())).tile_variant == 648
    assert errors(outputs[0].float().cpu().numpy(), want)[1] <= REL_L2


@pytest.mark.parametrize("dtype", ["float16", "bfloat16", "float32"])
def test_relu_after_the_second_contraction(oracle, dtype):
    # relu_out: the slot a fused activation layer lands in (chimera.graph_fusion)
    batch, M, N, K, L = 2, 200, 64, 40, 136
    A, B, C = oracle.make_gemm_chain_inputs(batch, M, N, K, L, dtype if dtype != "float32" else "float16", seed=9, std=0.25)
    want = np.maximum(oracle.bmm_chain_f64(A, B, C, inter="relu", round_mid=None if dtype == "float32" else dtype), 0.0)
    dev = "cuda:0"
    if dtype == "float32":
        a, b, c = (torch.from_numpy(x).to(dev) for x in (A, B, C))
    else:
        a, b, c = to_dev(A, dtype), to_dev(B, dtype), to_dev(C, dtype)
    for variant in ([0] if dtype == "float32" else variants(K, N, "KL")):
        f = torch.full((batch, M, N), float("nan"), device=dev, dtype=torch.float32)
        chain.run_bmm_chain(a, b, c, f, "relu", tile_variant=variant, relu_out=True)
        torch.cuda.synchronize()
        got = f.cpu().numpy()
        assert (got >= 0).all() and (got == 0).mean() > 0.2
        mx, rel = errors(got, want)
        assert mx <= MAX_ABS and rel <= REL_L2, (variant, mx, rel)
    with pytest.raises(NotImplementedError):  # no such slot behind the softmax chain
        chain.run_bmm_chain(a.half(), b.half(), c.half(), torch.empty(batch, M, N, device=dev, dtype=torch.float16),
                            "softmax", relu_out=True)
