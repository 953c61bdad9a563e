"""The matmul kernel of the tiled format, whichever way it comes by the rows that it multiplies: fragments that a pass packed, x lane by lane,
x (or the gradient's rows) through LDS.  Plans are made by hand, so that every form is reached at the sizes where it can go wrong."""
import pytest
import torch

from autogptq.tvm_amd import _lib, ops
from tests.parity_util import assert_tight, expected_weight, layer, to_dev
from tests.test_panel import assert_same_specials, with_weights


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


def forward_plan(M, K, N, bits, gs, row_tiles=1, split=1, wide=False):
    plan = _lib.select_tiled(130, K, N, bits, gs)
    assert plan.kernel == _lib.KERNEL_TILED
    plan.row_tiles, plan.waves_n, plan.waves_k = row_tiles, 2 if wide else 1, 4
    plan.m_blocks = plan.grid_z = -(-M // (32 * row_tiles))
    plan.grid_x = -(-(N // 32) // (4 if wide else 2))
    plan.k_chunk = -(-(-(-K // 64)) // (4 * split))
    plan.split_k = plan.grid_y = split
    plan.lds_bytes = 4 * row_tiles * 2 * 4096
    part = (split * M * N * 4 + 255) // 256 * 256 if split > 1 else 0
    plan.workspace_bytes = 16384 + part + split * 4 * plan.k_chunk * 4 * row_tiles * plan.m_blocks * 1024
    return plan


def transposed_plan(M, K, N, bits, gs, row_tiles=1, split=1, packed=False):
    """packed: empty row blocks behind the rows, more of them than workgroups find a place for their rows in LDS: the pass packs the rows, as it
    does for four row tiles."""
    plan = _lib.select_tiled_transposed(130, K, N, bits, gs)
    assert plan.kernel == _lib.KERNEL_TILED
    plan.row_tiles, plan.m_blocks = row_tiles, -(-M // (32 * row_tiles)) + (512 if packed and row_tiles < 4 else 0)
    plan.grid_z = plan.m_blocks
    plan.split_k = plan.grid_y = split
    plan.k_chunk = -(-(-(-N // 64)) // (4 * split))
    plan.lds_bytes = max(4 * row_tiles * 2 * 4096, 2 * 4 * plan.k_chunk * 256)
    part = (split * M * K * 4 + 255) // 256 * 256 if split > 1 else 0
    plan.workspace_bytes = 16384 + part + split * 4 * plan.k_chunk * 4 * row_tiles * plan.m_blocks * 1024
    return plan


def prepared(D):
    g = D["g_idx"] if D["desc_act"] else None
    return ops.tile_prepare(D["qweight"], D["qzeros"], D["scales"], g, D["bits"], D["group_size"])


def forward(D, tiles, plan, packed=False, x=None):
    """packed: with the channels' map, which a layer without an activation order has too (the identity): the pass runs."""
    maps = tiles[2:] if packed or D["desc_act"] else (None, None)
    return ops.gemm_tiled(D["x"] if x is None else x, tiles[0], tiles[1], *maps, None, D["bits"], D["group_size"], plan=plan)


def transposed(D, gy, xsrc, plan):
    qtile_t, szt = ops.tile_prepare_transposed(D["qweight"], D["qzeros"], D["scales"], xsrc, D["bits"], D["group_size"])
    return ops.gemm_tiled_transposed(gy, qtile_t, szt, xsrc, D["K"], D["bits"], D["group_size"], plan=plan)


# Half a block past K, whole blocks past it (alone, and behind ranges), both, neither: x is zero there, and an infinite weight of the last
# group (a scale of infinity, or a product beyond fp16) must not count
@pytest.mark.gpu
@pytest.mark.parametrize("bits", [2, 3, 4, 8])
@pytest.mark.parametrize("K", [32, 192, 352, 512, 832])
@pytest.mark.parametrize("scale", [60000.0, float("inf")])
def test_infinite_weights_of_the_last_group(dev, bits, K, scale):
    N, gs = 96, 32
    for desc_act in (False, True):
        L = layer(9100 + K, K, N, bits, gs, desc_act, M=130)
        L["x"] = L["x"].abs()
        with_weights(L, (5,), torch.full((K,), 3, dtype=torch.int32), 0.25)
        L["scales"][-1, 5] = scale
        W, D = expected_weight(L).float(), to_dev(L, dev)
        assert torch.isinf(W).sum() == gs and not torch.isnan(W).any()
        want, tiles = L["x"].float() @ W, prepared(D)
        for M, rt, split, wide in ((8, 1, 1, False), (8, 1, 2, False), (33, 1, 1, False), (33, 2, 3, False), (130, 4, 1, False),
                                   (130, 4, 2, False), (130, 4, 1, True), (130, 4, 2, True)):
            plan = forward_plan(M, K, N, bits, gs, rt, split, wide)
            for packed in (False, True):
                y = forward(D, tiles, plan, packed, x=D["x"][:M])
                assert_same_specials(y, want[:M], f"int{bits} K={K} act={desc_act} rows {M} tiles {rt} ranges {split} wide {wide} packed {packed}")


# the same for the gradient, whose reduction runs over the columns: one infinite weight in the last of them
@pytest.mark.gpu
@pytest.mark.parametrize("bits", [2, 3, 4, 8])
@pytest.mark.parametrize("N", [32, 192, 352, 512, 832])
def test_infinite_weights_of_the_last_column(dev, bits, N):
    K, gs, M = 256, 64, 130
    gy = torch.randn(M, N, generator=torch.Generator().manual_seed(7)).half()
    codes = torch.ones(K, dtype=torch.int32)
    codes[77] = 3                                       # 2 x 60000 does not fit fp16; the other weights of the column are zero
    for desc_act in (False, True):
        L = with_weights(layer(9200 + N, K, N, bits, gs, desc_act, M=M), (N - 1,), codes, 60000.0)
        W, D = expected_weight(L).float(), to_dev(L, dev)
        assert torch.isinf(W).sum() == 1 and not torch.isnan(W).any()
        want, xsrc = gy.float() @ W.t(), prepared(D)[2] if desc_act else None
        for rows, rt, split in ((8, 1, 1), (33, 1, 2), (33, 2, 1), (130, 4, 1), (130, 4, 3)):
            for packed in (False, True) if rt < 4 else (True,):
                gx = transposed(D, gy[:rows].to(dev), xsrc, transposed_plan(rows, K, N, bits, gs, rt, split, packed))
                assert_same_specials(gx, want[:rows], f"int{bits} N={N} act={desc_act} rows {rows} tiles {rt} ranges {split} packed {packed}")


# Up to 13 rows of a layer whose ranges cover K exactly x is read lane by lane, from 14 on and elsewhere through LDS, with a channels' map packed first:
# the same fragments and the same order of the sums, so the same bits
@pytest.mark.gpu
@pytest.mark.parametrize("bits", [2, 3, 4, 8])
@pytest.mark.parametrize("K,N,gs,split", [(256, 32, 32, 1), (768, 96, 64, 3), (1024, 416, 128, 2), (2048, 160, -1, 1), (4096, 96, 128, 8), (1056, 96, 32, 1)])
def test_rows_read_in_every_way_give_the_same_bits(dev, bits, K, N, gs, split):
    D = to_dev(layer(9300 + K, K, N, bits, gs, False, M=16), dev)
    tiles = prepared(D)
    want = D["x"].float().cpu() @ expected_weight({k: v.cpu() if torch.is_tensor(v) else v for k, v in D.items()}).float()
    for M in (1, 9, 12, 13, 14, 16):
        plan = forward_plan(M, K, N, bits, gs, 1, split)
        y, packed = forward(D, tiles, plan, x=D["x"][:M]), forward(D, tiles, plan, True, x=D["x"][:M])
        assert torch.equal(y, packed), f"int{bits} K={K} rows {M}"
        assert_tight(y, want[:M], f"int{bits} K={K} rows {M}")


# the gradient's rows through LDS and packed: the same bits
@pytest.mark.gpu
@pytest.mark.parametrize("bits", [2, 3, 4, 8])
@pytest.mark.parametrize("M,K,N,row_tiles,split", [(1, 64, 32, 1, 1), (31, 96, 352, 1, 1), (33, 160, 96, 1, 2), (64, 352, 1056, 2, 1), (65, 96, 2016, 2, 3),
                                                   (40, 320, 4096, 1, 4)])
def test_gradient_rows_in_both_ways_give_the_same_bits(dev, bits, M, K, N, row_tiles, split):
    gy = torch.randn(M, N, generator=torch.Generator().manual_seed(M)).half().to(dev)
    for desc_act in (False, True):
        D = to_dev(layer(9400 + N, K, N, bits, 32, desc_act), dev)
        xsrc = prepared(D)[2] if desc_act else None
        staged, packed = (transposed(D, gy, xsrc, transposed_plan(M, K, N, bits, 32, row_tiles, split, packed=p)) for p in (False, True))
        assert torch.equal(staged, packed), f"int{bits} act={desc_act}"


# the group of a lane block: groups of one block, of odd numbers of them, of half and of all of K
@pytest.mark.gpu
@pytest.mark.parametrize("bits", [3, 4])
@pytest.mark.parametrize("K,gs", [(1920, 32), (1920, 64), (1920, 96), (2080, 160), (4032, 224), (3936, 1312), (2112, 1056), (2016, -1)])
def test_groups_of_every_number_of_blocks(dev, bits, K, gs):
    N = 64
    D = to_dev(layer(9500 + K, K, N, bits, gs, True, M=40), dev)
    tiles, W = prepared(D), expected_weight({k: v.cpu() if torch.is_tensor(v) else v for k, v in D.items()}).float()
    for rt, split in ((1, 1), (2, 3)):
        y = forward(D, tiles, forward_plan(40, K, N, bits, gs, rt, split))
        assert_tight(y, D["x"].float().cpu() @ W, f"int{bits} K={K} groups of {gs} tiles {rt}")
