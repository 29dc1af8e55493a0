"""W8A16 dense linear: bf16 output against the fp32 closed form
C = A . (Q * s)^T (oracle ``w8a16_linear_f32``) on seeded inputs, to max_rel
and rel_fro <= 1e-2, at the benchmark shapes (K=4096, N in {4096, 1024,
16384}, M in {1, 64, 8192}), every split-K width, ragged M and N, and the
tiled packer against an independent numpy statement of its layout.

Every case runs twice: on the int8 weight as stored (row-major [N, K],
``w8a16_int8_gemm_into``) and on the load-time tiles (``prepare_int8_weight``,
``w8a16_prepared_gemm_into``); the two must give the same output bits.

Rows of C depend only on the same row of A, so M=8192 is checked on a seeded
subset of rows (the kernel still computes all of them).
"""

import numpy as np
import pytest
import torch

import oracle as O
from gaiban_lite_amd import ops, synthetic as S
from gaiban_lite_amd import weight_only_linear as L
from helpers import assert_moe_close, bf16_bits, to_np_f32

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def np_pack_int8(q: np.ndarray) -> np.ndarray:
    n, k = q.shape
    t = q.reshape(n // 16, 16, k // 64, 4, 16)          # strip, row, window, j, byte
    t = t.transpose(0, 2, 3, 1, 4)                       # strip, window, j, row, byte -> lane = 16j + row
    return np.ascontiguousarray(t).reshape(-1).view(np.uint8)


def run(m, n, k, *, split=None, seed=3, rows=None):
    print(f"[w8a16] M={m} N={n} K={k} split={split}", flush=True)
    q, s = S.make_int8_linear(n, k, seed=seed, device=DEV)
    a = torch.randn((m, k), device=DEV, generator=torch.Generator(DEV).manual_seed(seed + 100)).to(torch.bfloat16)
    prep = L.prepare_int8_weight(q, s)
    out = L.w8a16_linear(a, prep, split_k=split)
    raw = L.w8a16_linear(a, q, s, split_k=split)
    torch.cuda.synchronize()
    assert torch.equal(raw, out), "row-major and tiled weights differ"
    rows = np.arange(m) if rows is None else rows
    ref = O.w8a16_linear_f32(to_np_f32(a)[rows], q.cpu().numpy(), bf16_bits(s))
    err = assert_moe_close(to_np_f32(out)[rows], ref, what=f"M={m} N={n} split={split}")
    print(f"    {err}", flush=True)
    return out


def test_pack_int8_layout():
    q, _ = S.make_int8_linear(64, 256, seed=5, device=DEV)
    packed = ops.pack_int8(q)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(packed.cpu().numpy(), np_pack_int8(q.cpu().numpy()))


@pytest.mark.parametrize("n", [4096, 1024, 16384])
@pytest.mark.parametrize("m", [1, 64])
def test_decode_shapes(m, n):
    run(m, n, 4096)


@pytest.mark.parametrize("n", [4096, 1024, 16384])
def test_prefill_shapes_row_subset(n):
    rows = np.sort(np.random.default_rng(n).choice(8192, 96, replace=False))
    run(8192, n, 4096, rows=rows)


@pytest.mark.parametrize("split", [1, 2, 4, 8])
def test_every_split_width(split):
    out = run(64, 1024, 4096, split=split)
    base = run(64, 1024, 4096, split=1) if split != 1 else out
    # a different split only changes the fp32 summation order
    d = (out.float() - base.float()).abs().max().item()
    assert d <= 2e-2 * base.float().abs().max().item()


@pytest.mark.parametrize("m", [2, 3, 17, 33, 65, 100, 129])
@pytest.mark.parametrize("n,k", [(48, 256), (208, 384)])
def test_ragged_shapes(m, n, k):
    run(m, n, k)
    run(m, n, k, split=2)


def test_zero_rows_and_contract_errors():
    q, s = S.make_int8_linear(64, 256, device=DEV)
    prep = L.prepare_int8_weight(q, s)
    a = torch.empty((0, 256), dtype=torch.bfloat16, device=DEV)
    out = torch.empty((0, 64), dtype=torch.bfloat16, device=DEV)
    ops.w8a16_linear_into(a, prep.packed, prep.scale, out, None, n=64, split_k=1)
    ops.w8a16_linear_into(a, q, s, out, None, n=64, split_k=1)
    plan = L.make_gemm_plan(4, 64, 256, split_k=2)
    a = torch.zeros((4, 256), dtype=torch.bfloat16, device=DEV)
    out = torch.empty((4, 64), dtype=torch.bfloat16, device=DEV)
    ws = L.allocate_workspace(plan, DEV)
    with pytest.raises(ValueError):  # workspace shape
        L.w8a16_int8_gemm_into(a, q, s, out, torch.empty((1, 4, 64), dtype=torch.float32, device=DEV), plan=plan)
    with pytest.raises(ValueError):
        L.w8a16_prepared_gemm_into(a, prep, out, torch.empty((1, 4, 64), dtype=torch.float32, device=DEV),
                                   plan=plan)
    with pytest.raises(TypeError):  # activation dtype
        L.w8a16_int8_gemm_into(a.float(), q, s, out, ws, plan=plan)
    with pytest.raises(TypeError):  # weight dtype
        L.w8a16_int8_gemm_into(a, q.view(torch.uint8), s, out, ws, plan=plan)
    with pytest.raises(ValueError):  # weight shape
        L.w8a16_int8_gemm_into(a, q[:32], s, out, ws, plan=plan)
    with pytest.raises(TypeError):  # an int8 weight is not the checkpoint FP8 contract
        L.w8a16_gemm_into(a, q, s, out, ws, plan=plan)
    with pytest.raises(ValueError):
        L.make_gemm_plan(4, 64, 200)
    with pytest.raises(ValueError):
        L.make_gemm_plan(4, 64, 256, split_k=4)  # 2 K-blocks


def test_prefill_tile_with_explicit_split():
    """A whole-K prefill tile that sums a given K split in registers."""

    rows = np.sort(np.random.default_rng(7).choice(8192, 64, replace=False))
    run(8192, 4096, 4096, split=2, rows=rows)


@pytest.mark.parametrize("m,n,k,split", [(1, 4096, 4096, 8), (2, 1024, 4096, 2), (3, 16384, 4096, 4),
                                         (4, 4096, 1024, 8), (5, 1024, 4096, 4), (16, 4096, 4096, 2),
                                         (24, 1024, 4096, 8), (33, 4096, 4096, 4), (64, 1024, 4096, 8),
                                         (64, 16384, 4096, 4), (3, 208, 640, 4), (40, 208, 640, 4),
                                         (48, 4096, 4096, 8), (20, 208, 2048, 8)])
@pytest.mark.parametrize("fmt", ["int8", "fp8"])
def test_in_workgroup_split_matches_two_launch_reduction(m, n, k, split, fmt):
    """Up to 16 tokens a K split runs inside one workgroup (each wavefront
    one split's partial, summed through LDS in split order); from 17 on the
    partials go through the workspace and a reduce launch (up to 64 tokens
    with 4, 8 or 9 to 16 windows per split: weights straight to registers, the
    split's token rows in LDS), and the 128-token call sums them in registers
    where its tiles fill the chip (N=16384 here).  A row of C
    depends only on its row of A, and the split boundaries are the same, so
    the first m rows of a 128-token call with the same split must carry the
    same bits -- which pins the in-workgroup order of the additions.  Up to
    4 tokens with splits covering K exactly the activation rows go through
    LDS (M=1..4 here); ragged N and a last split shorter than the others
    included (K=640: 10 windows over 4 splits of 3)."""

    print(f"[w8a16 {fmt}] in-workgroup split M={m} N={n} K={k} split={split}", flush=True)
    gen = torch.Generator(DEV).manual_seed(m * 7 + split)
    a = torch.randn((128, k), device=DEV, generator=gen).to(torch.bfloat16)
    if fmt == "fp8":
        codes, scales = S.make_fp8_block_linear(n, k, seed=31, device=DEV)
        w, w_s = codes.view(torch.float8_e4m3fn), scales.view(torch.float8_e8m0fnu)
        prep = L.prepare_fp8_block_weight(codes, scales)
    else:
        w, w_s = S.make_int8_linear(n, k, seed=31, device=DEV)
        prep = L.prepare_int8_weight(w, w_s)
    small = L.w8a16_linear(a[:m].contiguous(), w, w_s, split_k=split)
    small_tiled = L.w8a16_linear(a[:m].contiguous(), prep, split_k=split)
    big = L.w8a16_linear(a, w, w_s, split_k=split)
    torch.cuda.synchronize()
    assert torch.equal(small.view(torch.int16), small_tiled.view(torch.int16))
    assert torch.equal(small.view(torch.int16), big[:m].view(torch.int16))


@pytest.mark.parametrize("m,n", [(385, 2064), (1000, 4080), (1000, 4112), (1500, 10000)])
@pytest.mark.parametrize("k,split", [(128, 1), (640, 1), (640, 2), (640, 4), (16384, 4), (16512, 8)])
@pytest.mark.parametrize("fmt", ["int8", "fp8"])
def test_many_token_tiles_carry_the_small_batch_bits(m, n, k, split, fmt):
    """Above 64 tokens one workgroup computes the whole K of its tile (64 x
    128, 128 x 128, 128 x 256 and, without a split, 256 x 256 tokens x
    channels for these shapes), adding each split's partial in split order:
    the rows carry the bits of a 40-token call with the same split, first and
    last tile included, for both weight layouts.  Ragged M and N, one K block
    and splits that end inside a K block (10 windows over 2 and 4 splits).  The
    two long K lie on the other side of the rule for the smaller grids, which run
    a workgroup per split there."""

    print(f"[w8a16 {fmt}] tiles M={m} N={n} K={k} split={split}", flush=True)
    gen = torch.Generator(DEV).manual_seed(m + split)
    a = torch.randn((m, k), device=DEV, generator=gen).to(torch.bfloat16)
    if fmt == "fp8":
        codes, scales = S.make_fp8_block_linear(n, k, seed=32, device=DEV)
        w, w_s = codes.view(torch.float8_e4m3fn), scales.view(torch.float8_e8m0fnu)
        prep = L.prepare_fp8_block_weight(codes, scales)
    else:
        w, w_s = S.make_int8_linear(n, k, seed=32, device=DEV)
        prep = L.prepare_int8_weight(w, w_s)
    big = L.w8a16_linear(a, w, w_s, split_k=split)
    tiled = L.w8a16_linear(a, prep, split_k=split)
    assert torch.equal(big.view(torch.int16), tiled.view(torch.int16))
    for row in (0, m - 40):
        small = L.w8a16_linear(a[row:row + 40].contiguous(), w, w_s, split_k=split)
        assert torch.equal(small.view(torch.int16), big[row:row + 40].view(torch.int16))


@pytest.mark.parametrize("k,split", [(2176, 8), (1152, 8)])
@pytest.mark.parametrize("fmt", ["int8", "fp8"])
def test_splits_past_the_end_of_k(k, split, fmt):
    """34 windows over 8 splits of 5 leave the last split empty, 18 over 8 of 3
    the last two: an empty split's partial is its zeros times the channel's
    scale, so a negative scale keeps the -0 of a zero row and an infinite or NaN
    scale makes the output NaN, above 64 tokens (the whole K in one workgroup)
    as in a 40-token call (a workgroup per split)."""

    m, n = 385, 4112
    print(f"[w8a16 {fmt}] empty splits M={m} N={n} K={k} split={split}", flush=True)
    a = torch.randn((m, k), device=DEV, generator=torch.Generator(DEV).manual_seed(k)).to(torch.bfloat16)
    a[::5] = 0.0
    if fmt == "fp8":
        codes, scales = S.make_fp8_block_linear(n, k, seed=34, device=DEV)
        w, w_s = codes.view(torch.float8_e4m3fn), scales.view(torch.float8_e8m0fnu)
    else:
        w, w_s = S.make_int8_linear(n, k, seed=34, device=DEV)
        w_s[::3] *= -1.0
        for c, v in ((16, float("inf")), (33, float("-inf")), (4100, float("nan"))):
            w_s[c] = v
    big = L.w8a16_linear(a, w, w_s, split_k=split)
    for row in (0, m - 40):
        small = L.w8a16_linear(a[row:row + 40].contiguous(), w, w_s, split_k=split)
        part = big[row:row + 40]
        assert torch.equal(small.isnan(), part.isnan())
        bits = torch.where(small.isnan(), torch.zeros_like(small), small).view(torch.int16)
        assert torch.equal(bits, torch.where(part.isnan(), torch.zeros_like(part), part).view(torch.int16))


@pytest.mark.parametrize("m", [17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("n,k,split", [(14352, 4096, 4), (2000, 2304, 4), (2000, 1152, 2),
                                       (14352, 3712, 4), (14352, 3200, 4), (2000, 5376, 8), (2000, 4480, 8),
                                       (2000, 3456, 4), (1008, 896, 1)])
@pytest.mark.parametrize("fmt", ["int8", "fp8"])
def test_nine_to_sixteen_windows_carry_the_larger_batch_bits(m, n, k, split, fmt):
    """17 to 64 tokens with 9 to 16 windows per split, on both sides of the rule
    for weights straight to registers: eight wavefronts per workgroup at N=14352
    (ragged last tile; row-major weights, the tiles and 13 windows above 32 tokens
    run the other kernel), four at N=2000 and 1008, 32, 48 and 64 token rows, last
    splits of fewer windows (K=3712: 15, 15, 15, 13; 5376: 7 x 11 and 7; 4480: 7 x
    9 and 7).  A row depends only on its own activations and the splits are the
    same, so the bits are those of a 128-token call, which runs another kernel."""

    test_in_workgroup_split_matches_two_launch_reduction(m, n, k, split, fmt)


@pytest.mark.parametrize("split", [2, 4, 8, 16])
@pytest.mark.parametrize("m,n", [(17, 16), (64, 2048), (61, 2176), (64, 12288), (63, 12496)])
def test_split_reduction_counts_and_sizes(m, n, split):
    """The reduce launch for each number of splits that the library takes (4 and
    8 have their own code, 2 and 16 the general one; plans stop at 8) and on both
    sides of its change of workgroup size (64 x 2048 outputs) and of its return to
    the general code (64 x 12288), against the float64 sum of the workspace's partials rounded once: the fp32 additions
    differ from it by at most split - 1 roundings of 2^-24 of the sum of
    magnitudes (1.01 covers their second order), bf16 by 2^-8 of the value."""

    k = 2048
    print(f"[w8a16 fp8] reduce launch M={m} N={n} split={split}", flush=True)
    a = torch.randn((m, k), device=DEV, generator=torch.Generator(DEV).manual_seed(m + split)).to(torch.bfloat16)
    codes, scales = S.make_fp8_block_linear(n, k, seed=33, device=DEV)
    ws = torch.full((split, m, n), float("nan"), dtype=torch.float32, device=DEV)
    out = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
    ops.w8a16_fp8_linear_into(a, codes, scales, out, ws, n=n, split_k=split)
    torch.cuda.synchronize()
    partial = ws.double()
    ref = partial.sum(0)
    bound = ref.abs() * 2.0 ** -8 + partial.abs().sum(0) * (1.01 * (split - 1) * 2.0 ** -24)
    assert bool(((out.double() - ref).abs() <= bound).all())
