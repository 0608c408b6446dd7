"""A token's output does not depend on the other tokens of the call: the first rows of a
batch give the same bits as a smaller batch of those rows, on each path (the reference's
check of its fused decode kernel, tests/test_fused_moe.py:107, "a row's output is
independent of the row count").

Within one path (decode, tiled, prefill) the per-row arithmetic is fixed: the router's dot
products, the top-k, each expert projection's K order and the combine are per token, so
the comparison is bitwise. The router GEMM of the tiled and prefill paths sums every logit
in one fixed order at every batch size: its K-quarter kernel (the block's from 5 tokens on, with
wide routers of short rows from 9, to 384), its split kernel (otherwise below 768 tokens, in
three tile configurations switching at 128 and 384) and its LDS-tiled DMA kernel (from 768)
give the same bits. 800 -> 700, 1024 -> 600 and 2048 -> 100 cross from the DMA kernel to
the split one (1024 -> 600 and 800 -> 700 within the prefill GEMM tiles; 2048 -> 100 also
crosses from the prefill GEMM tiles to the tiled expert GEMM, so there only the routing is
bitwise), 512 -> 300 from the split kernel to K quarters. So the logits themselves
are bitwise too. Across
paths the fp32 summation order of a projection differs and only the bf16 tolerance applies
(tested elsewhere)."""

from __future__ import annotations

import pytest
import torch

from oracle import moe_oracle as orc

pytestmark = pytest.mark.gpu

BF16 = torch.bfloat16


@pytest.fixture(scope="module")
def mlp(dev):
    import __graft_entry__

    return __graft_entry__._mlp_from_weights(orc.make_weights(2048, 256, 512, 512, seed=31), dev)


@pytest.mark.parametrize("big,small,decode", [(4, 1, True), (4, 3, True), (16, 9, True),
                                              (16, 5, False), (100, 64, False),
                                              (255, 17, False), (512, 300, False), (300, 129, False),
                                              (1536, 1024, False),
                                              (4096, 2048, False), (1100, 900, False),
                                              (800, 700, False), (1024, 600, False),
                                              (2048, 100, False), (8192, 4096, False)])
def test_leading_rows_match_smaller_batch(pkg, dev, mlp, big, small, decode):
    print(f"row independence {big} -> {small} decode={decode}", flush=True)
    g = torch.Generator().manual_seed(big + small)
    x = torch.randn(big, 2048, generator=g).to(BF16).to(dev)
    r = torch.randn(big, 2048, generator=g).to(BF16).to(dev)
    a, ia, wa, la = pkg.block.moe(x, mlp, 8, decode=decode, residual=r, return_routing=True)
    b, ib, wb, lb = pkg.block.moe(x[:small].contiguous(), mlp, 8, decode=decode,
                                  residual=r[:small].contiguous(), return_routing=True)
    torch.cuda.synchronize()
    assert torch.equal(la[:small], lb), "router logits depend on the batch"
    assert torch.equal(ia[:small], ib) and torch.equal(wa[:small], wb)
    # the experts' GEMM path changes above 512 tokens (tiled -> prefill tiles), with its own
    # fp32 summation order: across that boundary only the routing is compared
    if (big > 512) == (small > 512):
        assert torch.equal(a[:small], b)


@pytest.mark.parametrize("H,E", [(512, 256), (1024, 256), (512, 16)])
def test_leading_rows_match_across_router_kernels(pkg, dev, H, E):
    """Routers of other widths take the split kernel up to 4 or, wide ones of short rows, 8 tokens and
    K quarters above: the same logits and outputs, bit for bit, on both sides (decode=True: without
    it the products' rounding changes above 16 tokens)."""
    print(f"row independence across router kernels H={H} E={E}", flush=True)
    import __graft_entry__

    mlp = __graft_entry__._mlp_from_weights(orc.make_weights(H, E, 128, 128, seed=7), dev)
    x = torch.randn(20, H, generator=torch.Generator().manual_seed(H + E)).to(BF16).to(dev)
    a, ia, wa, la = pkg.block.moe(x, mlp, 8, decode=True, return_routing=True)
    for n in (16, 9, 8, 5):
        b, ib, wb, lb = pkg.block.moe(x[:n].contiguous(), mlp, 8, decode=True, return_routing=True)
        torch.cuda.synchronize()
        assert torch.equal(la[:n], lb) and torch.equal(ia[:n], ib) and torch.equal(wa[:n], wb)
        assert torch.equal(a[:n], b)


@pytest.mark.parametrize("big,small,I", [(1024, 600, 512), (1100, 900, 512), (4096, 2048, 512),
                                         (6000, 4096, 512), (8192, 5000, 512), (132000, 4096, 512),
                                         (1100, 900, 1024), (1024, 600, 1024)])
def test_leading_rows_match_smaller_batch_fp8_prefill(pkg, dev, big, small, I):
    """The e4m3 prefill kernels: a row's bits do not depend on the batch either where its rows
    fall into another part or block count of a tile, where the batch takes the other kernel (above
    128 rows per expert on average: 4096 tokens; with an intermediate of 1024 down below 32, 1024
    tokens, and gate_up below 24), or where the outputs of the experts are past 4 GiB (131072 tokens)."""
    print(f"fp8 row independence {big} -> {small} I={I}", flush=True)
    E, H, k = 256, 2048, 8
    g = torch.Generator(device=dev).manual_seed(big + small)

    def weight(*shape):
        return (torch.randn(*shape, generator=g, device=dev) * 100).clamp(-448, 448).to(
            torch.float8_e4m3fn)

    gu, dn = weight(E, 2 * I, H), weight(E, H, I)
    scales = dict(gate_up_scale=torch.rand(E, 2 * I, generator=g, device=dev) * 4e-4,
                  down_scale=torch.rand(E, H, generator=g, device=dev) * 4e-4)
    x = torch.randn(big, H, generator=g, device=dev).to(BF16)
    idx = torch.rand(big, E, generator=g, device=dev).topk(k, dim=1).indices
    w = torch.full((big, k), 0.125, dtype=BF16, device=dev)
    a = pkg.ops.moe_prefill(x, idx, w, gu, dn, **scales)[:small].clone()
    b = pkg.ops.moe_prefill(x[:small].contiguous(), idx[:small].contiguous(),
                            w[:small].contiguous(), gu, dn, **scales)
    torch.cuda.synchronize()
    assert torch.isfinite(a).all() and a.float().abs().mean() > 1e-3
    assert torch.equal(a, b)
