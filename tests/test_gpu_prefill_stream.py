"""The prefill kernels (e4m3 streaming, e4m3 and bf16 staged through LDS) at the edges of their
tiles: every 16-token block count they are compiled for with the rows one below, at and one
above a block boundary, parts of a larger table tile, each ring depth of the streaming kernel (K
of 256, 384, 512, 768 and 1024), the K that the staged e4m3 kernel takes instead (64, 128, 192) and
experts without rows; above 128 rows per expert on average, and for gate_up below 16 to 24 (K / 32
where K is no power of two) and down below K / 32 (K above 512), the staged e4m3 kernel; down with one and
with two row blocks per workgroup.

Tolerance: the results are bf16 roundings of fp32 sums of K bf16 products; the reference sums
in float64 and rounds at the same points, so a rounded value differs by one bf16 ulp (at most
2^-7 of it) only where its sum lies within the fp32 error of a rounding boundary. Down: one such
rounding, 2^-7. gate_up: those of gate (which silu magnifies by |1 + x (1 - sigmoid(x))|, at most
8 for the |x| <= 9 met here), silu, up and product: 11 * 2^-7; and 2^-16 of the row's largest
value for sums that cancel. Few values meet a boundary: the mean difference is at most 2^-11 of
the mean value."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.fixture(scope="module")
def pkg():
    import __graft_entry__

    return __graft_entry__.load_package()


def _routing(counts, k):
    """top_k_index [T, 1] giving expert e exactly counts[e] pairs, in a shuffled order."""
    ids = torch.cat([torch.full((c,), e) for e, c in enumerate(counts)])
    g = torch.Generator().manual_seed(len(ids))
    return ids[torch.randperm(len(ids), generator=g)].reshape(-1, k).long()


def _bf(x):
    return x.to(BF16).double()


def _close(got, ref, rel):
    got, ref = got.double().cpu(), ref.cpu()
    bound = rel * ref.abs() + 2.0**-16 * ref.abs().amax(-1, keepdim=True)
    assert torch.isfinite(got).all()
    diff = (got - ref).abs()
    assert (diff <= bound).all(), (diff - bound).max().item()
    assert diff.mean() <= 2.0**-11 * ref.abs().mean()


def _weights(E, H, I, fp8, pkg, dev):
    g = torch.Generator().manual_seed(E + H + I)
    gu = (torch.randn(E, 2 * I, H, generator=g) * 0.05).to(BF16)
    dn = (torch.randn(E, H, I, generator=g) * 0.05).to(BF16)
    if not fp8:
        return (gu.to(dev), None, dn.to(dev), None), (gu.double(), dn.double())
    (qg, sg), (qd, sd) = pkg.fp8.quantize_rows(gu), pkg.fp8.quantize_rows(dn)
    deq = [q.float().double() * s.double()[..., None] for q, s in ((qg, sg), (qd, sd))]
    return tuple(t.to(dev) for t in (qg, sg, qd, sd)), deq


# rows per expert around the block counts (2, 4 / 4, 6, 8, 10 blocks of 16) and past a tile
SMALL = [0, 1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 1, 130]
LARGE = [0, 79, 80, 81, 95, 96, 97, 127, 128, 129, 159, 160, 161, 3, 320, 63]


# more than 128 rows per expert on average: edges of whole 256-row tiles and of the last one
MANY = [0, 255, 256, 257, 511, 512, 513, 1, 272, 290]
# fewer than 16 rows per expert on average
FEW = [0, 1, 2, 5, 15, 16, 17, 31, 3, 33, 0, 0, 7, 1, 0, 0]


SHAPES = [(256, 128, True), (256, 384, True), (768, 128, True), (1024, 256, True), (512, 512, True),
          (256, 1024, True), (512, 128, False), (768, 256, False), (256, 128, False)]
# hidden sizes that the whole call takes on 64-row tiles
GROUPED_ONLY = [(64, 128, True), (192, 128, True)]


@pytest.mark.parametrize("H,I,fp8,counts,bm", [
    (*shape, counts, bm) for bm in (256, None) for shape in SHAPES + (GROUPED_ONLY if bm else [])
    for counts in (SMALL, LARGE, MANY) + ((FEW,) if bm else ())])
def test_prefill_stream_tiles(pkg, H, I, fp8, counts, bm):
    """bm None: the whole routed-experts call with its own tile size (more than 512 tokens);
    256: the grouped operations on a table of 256-row tiles."""
    print(f"prefill stream H={H} I={I} fp8={fp8} rows<= {max(counts)} bm={bm}", flush=True)
    dev = torch.device("cuda")
    E, T = len(counts), sum(counts)
    (gu, gus, dn, dns), (gu64, dn64) = _weights(E, H, I, fp8, pkg, dev)
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, H, generator=g).to(BF16)
    idx = _routing(counts, 1)
    act = torch.zeros(T, I, dtype=torch.float64)
    y = torch.zeros(T, H, dtype=torch.float64)
    for e in range(E):
        t = torch.where(idx[:, 0] == e)[0]
        gate, up = _bf(x[t].double() @ gu64[e][:I].T), _bf(x[t].double() @ gu64[e][I:].T)
        act[t] = _bf(_bf(gate * torch.sigmoid(gate)) * up)
        y[t] = act[t] @ dn64[e].T
    if bm is None:
        # weights of 1: the combine passes y through
        out = pkg.ops.moe_prefill(x.to(dev), idx.to(dev), torch.ones(T, 1, dtype=BF16, device=dev),
                                  gu, dn, gate_up_scale=gus, down_scale=dns)
        torch.cuda.synchronize()
        # act off in places as above: its effect on y is at most that share of sum |act w|
        bound = torch.zeros(T, H, dtype=torch.float64)
        for e in range(E):
            t = torch.where(idx[:, 0] == e)[0]
            bound[t] = act[t].abs() @ dn64[e].abs().T
        diff = (out.double().cpu() - _bf(y)).abs()
        assert (diff <= 2.0**-7 * y.abs() + 11 * 2.0**-7 * bound).all()
        assert diff.mean() <= 2.0**-10 * y.abs().mean()
        return
    sp = pkg.ops.sort_pairs(idx.to(dev), E, bm=bm)
    got = pkg.ops.grouped_gate_up(x.to(dev), 1, gu, sp, gus)
    order = sp.order.long().cpu()
    torch.cuda.synchronize()
    _close(got, act[order], 11 * 2.0**-7)
    got_y = pkg.ops.grouped_down(act[order].to(BF16).to(dev), T, 1, dn, sp, dns)
    torch.cuda.synchronize()
    _close(got_y, _bf(y), 2.0**-7)


@pytest.mark.parametrize("K", [256, 512, 640, 1024])
@pytest.mark.parametrize("E,H", [(130, 512), (100, 768), (64, 1056)])
def test_prefill_stream_down_row_blocks(pkg, E, H, K):
    """e4m3 down with enough experts for two row blocks per workgroup, whole pairs of blocks, an odd
    block (H = 768) and a partial last one (1056), for each form of the walk over K (two phases in
    LDS: 512)."""
    print(f"prefill stream down row blocks E={E} H={H} K={K}", flush=True)
    dev = torch.device("cuda")
    counts = [(SMALL + LARGE)[e % 32] for e in range(E)]
    T = sum(counts)
    assert 32 * E <= T <= 128 * E
    g = torch.Generator(device=dev).manual_seed(E + K)
    w = (torch.randn(E, H, K, generator=g, device=dev) * 100).clamp(-448, 448).to(torch.float8_e4m3fn)
    scale = torch.rand(E, H, generator=g, device=dev) * 4e-4
    act = torch.randn(T, K, generator=g, device=dev).to(BF16)
    idx = _routing(counts, 1).to(dev)
    sp = pkg.ops.sort_pairs(idx, E, bm=256)
    got = pkg.ops.grouped_down(act, T, 1, w, sp, scale)
    order = sp.order.long()
    want = torch.empty(T, H, dtype=torch.float64, device=dev)
    r = 0
    for e in range(E):
        rows = slice(r, r + counts[e])
        want[order[rows]] = act[rows].double() @ (w[e].double() * scale[e].double()[:, None]).T
        r += counts[e]
    torch.cuda.synchronize()
    _close(got, _bf(want).cpu(), 2.0**-7)


@pytest.mark.parametrize("K", [32, 96, 160, 224])
def test_prefill_bf16_half_chunk(pkg, K):
    """bf16 rows of an odd multiple of 32 on 256-row tiles, with a shared expert of the same and of
    another length in the launch: K is walked in chunks of 64, whose last one is a half."""
    print(f"prefill half chunk K={K}", flush=True)
    dev = torch.device("cuda")
    counts, N, IS = [0, 1, 17, 255, 256, 257, 300], 128, 128
    E, T = len(counts), sum(counts)
    g = torch.Generator().manual_seed(K)

    def rnd(*shape):
        return (torch.randn(*shape, generator=g) * 0.25).to(BF16)

    def act(x, gate, up):
        gt, u = _bf(x @ gate.double().T), _bf(x @ up.double().T)
        return _bf(_bf(gt * torch.sigmoid(gt)) * u)

    idx = _routing(counts, 1)
    sp = pkg.ops.sort_pairs(idx.to(dev), E, bm=256, shared=True)
    order = sp.order.long().cpu()
    expert = idx[order, 0]
    # gate_up: hidden K
    x, gu, sg, su = rnd(T, K), rnd(E, 2 * N, K), rnd(IS, K), rnd(IS, K)
    ref = torch.cat([act(x[order][expert == e].double(), gu[e, :N], gu[e, N:]) for e in range(E)])
    got, got_sh = pkg.ops.grouped_gate_up(x.to(dev), 1, gu.to(dev), sp,
                                          shared=(sg.to(dev), su.to(dev)))
    torch.cuda.synchronize()
    _close(got, ref, 11 * 2.0**-7)
    _close(got_sh, act(x.double(), sg, su), 11 * 2.0**-7)
    # down: intermediate K, the shared expert's K and 128
    for Ks in (K, 128):
        a, dn, sd, ash = rnd(T, K), rnd(E, N, K), rnd(N, Ks), rnd(T, Ks)
        y = torch.empty(T, N, dtype=torch.float64)
        for e in range(E):
            y[order[expert == e]] = a[expert == e].double() @ dn[e].double().T
        got, got_sh = pkg.ops.grouped_down(a.to(dev), T, 1, dn.to(dev), sp,
                                           shared=(sd.to(dev), ash.to(dev)))
        torch.cuda.synchronize()
        _close(got, _bf(y), 2.0**-7)
        _close(got_sh, _bf(ash.double() @ sd.double().T), 2.0**-7)


@pytest.mark.parametrize("fp8,rows", [(False, 20), (True, 20), (True, 129)])
def test_prefill_stream_silu_range(pkg, fp8, rows):
    """gate_up's SiLU over its whole range: one gate value per expert (e4m3: by the row's scale),
    up = 1, a down row that passes act[0] through. Against float64 within one bf16 ulp (2^-7 of
    the value); below x = -88.7, where exp(-x) is past float32, the value is under 3e-37 and may
    come out as 0; infinities and NaN as torch's."""
    print(f"silu range fp8={fp8} rows={rows}", flush=True)
    dev = torch.device("cuda")
    inf = float("inf")
    vals = [0.0, 1e-30, -1e-30, 0.5, -0.5, 1.0, -1.0, 3.0, -3.0, 7.5, -7.5, 20.0, -20.0, 44.25, -44.5,
            60.0, -60.0, -80.0, -86.0, -87.0, 87.5, -87.5, -88.0, 88.5, -88.5, 89.0, -89.0, -95.0,
            300.0, -300.0, 1e8, -1e8, 1e20, -1e20, 3e38, inf, -inf, float("nan")]
    E, T, H, I = len(vals), rows * len(vals), 256, 128
    v = torch.tensor(vals, dtype=torch.float64).to(BF16)
    gu = torch.zeros(E, 2 * I, H, dtype=BF16)
    gu[:, 0, 0] = 1.0 if fp8 else v
    gu[:, I, 0] = 1.0
    dn = torch.zeros(E, H, I, dtype=BF16)
    dn[:, 0, 0] = 1.0
    scales = {}
    if fp8:
        gu, dn = gu.to(torch.float8_e4m3fn), dn.to(torch.float8_e4m3fn)
        gus = torch.ones(E, 2 * I)
        gus[:, 0] = v.float()
        scales = dict(gate_up_scale=gus.to(dev), down_scale=torch.ones(E, H, device=dev))
    x = torch.zeros(T, H, dtype=BF16)
    x[:, 0] = 1.0
    idx = _routing([rows] * E, 1)
    out = pkg.ops.moe_prefill(x.to(dev), idx.to(dev), torch.ones(T, 1, dtype=BF16, device=dev),
                              gu.to(dev), dn.to(dev), **scales)
    torch.cuda.synchronize()
    got = out[:, 0].double().cpu()
    v64 = v.double()
    ref = (v64 * torch.sigmoid(v64))[idx[:, 0]]
    for g, r, e in zip(got.tolist(), ref.tolist(), idx[:, 0].tolist()):
        if r != r:
            assert g != g, vals[e]
        elif r == inf:
            assert g == inf, vals[e]
        else:
            assert abs(g - r) <= (abs(r) if vals[e] < -88.7 else 2.0**-7 * abs(r)), (vals[e], g, r)
