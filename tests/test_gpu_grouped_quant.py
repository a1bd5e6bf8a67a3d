"""Grouped quantizer in one launch: the group boundaries inside the table search (empty groups at every place, one group, more
groups than the table holds) against the per-group oracle; row padding at the edges of a lane's pieces."""
import numpy as np
import pytest
import torch

import mdy_triton_amd as m
from mdy_triton_amd.megatron_patchs import dpsk_grouped_linear as PG
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("splits,N,strided", [([256], 256, False), ([0, 256, 0, 0, 512, 0], 512, False), ([256, 0], 256, True),
                                              ([512, 256, 256], 7168, False), ([0, 0], 256, False), ([256] * 3 + [0] * 300, 256, False),
                                              ([0] * 256 + [256], 256, False), ([256] + [0] * 270 + [256], 256, False),
                                              ([0] * 127 + [512, 256], 256, True), ([256] * 130, 256, False)])
def test_group_boundaries(splits, N, strided):
    x = torch.randn(sum(splits), N, generator=torch.Generator().manual_seed(len(splits))).bfloat16()
    xd = x.cuda()
    if strided:
        xd = xd.t().contiguous().t()
    y, s, yt, st = m.group_per_token_cast_to_fp8(xd, splits)
    assert len(yt) == len(st) == len(splits)
    row = 0
    for mg, a, b in zip(splits, yt, st):
        assert a.shape == (N, mg) and a.is_contiguous() and b.shape == (N, mg // 128)
        if mg:
            ry, rs, ryt, rst = O.per_token_cast_to_fp8(x[row:row + mg], True)
            for got, ref in ((y[row:row + mg], ry), (s[row:row + mg], rs), (a, ryt), (b, rst)):
                assert np.array_equal(got.cpu().contiguous().view(torch.uint8).numpy(), ref.contiguous().view(torch.uint8).numpy())
        row += mg


@pytest.mark.parametrize("wrapper", [False, True])       # the native call and the wrapper
def test_every_group_is_a_tensor_of_its_own(wrapper):
    """One group's copy changed or given up: the others can still be saved for a backward pass, and its memory is free."""
    from mdy_triton_amd.megatron_patchs.manger import CustomManger

    class Splits(tuple):      # what the native call leaves to the wrapper
        pass

    splits = (Splits if wrapper else list)([4096, 256, 512])
    x = torch.randn(sum(splits), 2048, device="cuda").bfloat16()
    _, _, yt, st = m.group_per_token_cast_to_fp8(x, splits)

    class Keep(torch.autograd.Function):
        @staticmethod
        def forward(ctx, a, *saved):
            ctx.save_for_backward(*saved)
            return a * 2

        @staticmethod
        def backward(ctx, g):
            assert len(ctx.saved_tensors) == 4
            return (g * 2,) + (None,) * 4

    a = torch.ones(1, requires_grad=True, device="cuda")
    out = Keep.apply(a, yt[1], yt[2], st[1], st[2])
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    CustomManger.clear_tensor_data(yt[0], st[0])
    assert before - torch.cuda.memory_allocated() >= 4096 * 2048
    out.backward()
    assert a.grad.item() == 2


@pytest.mark.parametrize("H", [8, 504, 512, 520, 2040, 2048, 2056, 3, 255, 257])      # bf16: around 64 and 256 pieces of 16, 2 and 1 bytes
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.uint8])
def test_padding_at_piece_edges(H, dtype):
    splits = [5, 0, 256, 257, 1]
    x = torch.randint(0, 200, (sum(splits), H), generator=torch.Generator().manual_seed(H)).to(dtype).cuda()
    p = PG.pad_groups(x, splits)
    row = slot = 0
    for mg in splits:
        pm = (mg + 255) // 256 * 256
        assert torch.equal(p[slot:slot + mg], x[row:row + mg]) and not p[slot + mg:slot + pm].any()
        row, slot = row + mg, slot + pm
    assert torch.equal(PG.unpad_groups(p, splits), x)


@pytest.mark.parametrize("G,N,K", [(2, 128, 256), (65, 130, 200), (3, 300, 264)])      # 65: more than one launch holds
@pytest.mark.parametrize("normal,transpose", [(True, False), (True, True), (False, True)])
def test_weight_list(G, N, K, normal, transpose):
    g = torch.Generator().manual_seed(G)
    ws = [(torch.randn(N, K, generator=g) * (i + 1)).bfloat16() for i in range(G)]
    wd = [w.cuda() if i != 1 else w.cuda().t().contiguous().t() for i, w in enumerate(ws)]      # one of other strides
    for got, ref in zip(m.per_block_cast_to_fp8(wd, normal, transpose), O.per_block_cast_to_fp8(ws, normal, transpose)):
        assert got.shape == ref.shape
        assert np.array_equal(got.cpu().view(torch.uint8).numpy(), ref.view(torch.uint8).numpy())
