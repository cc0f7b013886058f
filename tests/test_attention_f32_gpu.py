"""The FP32 matrix-core attention against the formula in 64 bits: tile edges of
the 16-key tiles and 16-row blocks, key splits, windows, trees, sinks, gates,
strides and alignments that change the kernel, rows no query may touch, and a
caller without a workspace.

The bound: each score is a sum of c products (relative error of the sum at
most c ulp / 2 of the products' sum, in practice below 8 ulp of |s| <= 6 at
these inputs), a weight's relative error is that of its score's difference, and
the output is a convex combination of values below 5: 2e-6 of the largest
output, four times under the reference's FP32 criterion of 1e-5."""

import ctypes

import pytest
import torch

from wpt_amd import _lib, kernels

pytestmark = pytest.mark.gpu
BOUND = 2e-6


def formula(q, k, v, visible, scale, sink=None):
    """visible (B, T, N)"""
    s = torch.einsum("bthc,bnc->bthn", q.double(), k.double()) * scale
    s = s.masked_fill(~visible[:, :, None], -float("inf"))
    if sink is not None:
        s = torch.cat([s, sink.double()[None, None, :, None].expand(*s.shape[:3], 1)], -1)
    lse = torch.logsumexp(s, -1)
    p = torch.softmax(s, -1).nan_to_num(0.0)
    if sink is not None:
        p = p[..., :-1]
    seen = torch.where(visible.any(1)[..., None], v.double(), 0.0)  # a row nobody sees may hold anything
    return torch.einsum("bthn,bnc->bthc", p, seen), lse


def causal(positions, N, window=0):
    n = torch.arange(N)
    seen = n <= positions[..., None]
    return seen & (n > positions[..., None] - window) if window else seen


def inputs(B, T, H, c, N, seed=0):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(B, T, H, c, generator=g)
    table = torch.randn(B, N, 2 * c, generator=g)
    return g, q, table[..., :c], table[..., c:], (N - T + torch.arange(T)).expand(B, T).contiguous()


def check(got, expected):
    assert torch.isfinite(got).all()
    error = float((got.cpu().double() - expected).abs().max() / expected.abs().max())
    assert error < BOUND, error


@pytest.mark.parametrize("B,T,H,c,N,splits", [
    (1, 1, 1, 64, 1, 0), (2, 1, 4, 64, 16, 0), (1, 5, 4, 64, 17, 0), (3, 5, 4, 128, 63, 0), (8, 5, 4, 64, 1029, 0),
    (1, 5, 16, 128, 300, 0), (2, 3, 16, 128, 257, 3), (1, 9, 16, 64, 130, 0), (1, 9, 8, 128, 129, 64),
    (2, 33, 8, 64, 200, 0), (1, 200, 4, 64, 200, 1), (16, 2, 16, 128, 65, 2), (1, 4, 17, 64, 640, 1)])
def test_chain(device, B, T, H, c, N, splits):
    print(f"fp32 chain B={B} T={T} H={H} c={c} N={N} splits={splits}", flush=True)
    g, q, k, v, positions = inputs(B, T, H, c, N)
    sink = torch.randn(H, generator=g)
    table = torch.cat([k, v], -1).to(device)
    for use in (None, sink):
        expected, lse = formula(q, k, v, causal(positions, N), c ** -0.5, use)
        got, got_lse = kernels.verify_attention(q.to(device), table[..., :c], table[..., c:], positions.to(device),
                                                c ** -0.5, sink=use, lse=True, splits=splits)
        check(got, expected)
        assert float((got_lse.cpu() - lse).abs().max()) < 4e-6


@pytest.mark.parametrize("c", [64, 128])
def test_positions_of_any_kind(device, c):
    """Before the text, past the table, out of order; a window; a scale below 0."""
    g, q, k, v, _ = inputs(2, 6, 4, c, 90, seed=1)
    positions = torch.tensor([[-3, 0, 200, 17, 16, 89], [31, 5, -1, 88, 47, 48]])
    kd, vd, pd = k.to(device), v.to(device), positions.to(device)
    for window, scale in ((0, c ** -0.5), (20, c ** -0.5), (0, -0.07)):
        seen = causal(positions, 90, window)
        expected, lse = formula(q, k, v, seen, scale)
        got, got_lse = kernels.verify_attention(q.to(device), kd, vd, pd, scale, window=window, lse=True)
        none = ~seen.any(-1)
        assert (got.cpu()[none] == 0).all() and (got_lse.cpu()[none] == -float("inf")).all()
        check(got, expected.masked_fill(none[..., None, None], 0.0))
        assert float((got_lse.cpu() - lse)[~none].abs().max()) < 4e-6


@pytest.mark.parametrize("B,M,H,c,prefix", [(2, 31, 4, 64, 100), (1, 63, 16, 128, 33), (8, 7, 4, 64, 16)])
def test_tree(device, B, M, H, c, prefix):
    g, q, k, v, _ = inputs(B, M, H, c, prefix + M, seed=2)
    parents = [-1] + [int(torch.randint(0, i, (1,), generator=g)) for i in range(1, M)]
    seen = torch.zeros(M, prefix + M, dtype=torch.bool)
    seen[:, :prefix] = True
    for i, parent in enumerate(parents):
        if parent >= 0:
            seen[i, prefix:] = seen[parent, prefix:]
        seen[i, prefix + i] = True
    expected, _ = formula(q, k, v, seen.expand(B, -1, -1), c ** -0.5)
    base = torch.full((B,), prefix, device=device)
    check(kernels.tree_attention(q.to(device), k.to(device), v.to(device), base, parents, c ** -0.5), expected)


@pytest.mark.parametrize("T,past", [(1, 3), (5, 300), (129, 513)])
def test_a_gated_window_over_a_ring(device, T, past):
    B, H, c, window = 3, 4, 64, 128
    g, q, k, v, positions = inputs(B, T, H, c, past + T, seed=3)
    sink, gate = torch.randn(H, generator=g), torch.randn(B, T, H * c, generator=g)
    ring = torch.zeros(B, 256, 2 * c)
    held = torch.arange(max(0, past + T - 256), past + T)
    ring[:, held % 256] = torch.cat([k, v], -1)[:, held]
    expected, _ = formula(q, k, v, causal(positions, past + T, window), c ** -0.5, sink)
    got = kernels.ring_attention(q.to(device), ring.to(device), positions.to(device), c ** -0.5, window,
                                 sink.to(device), gate=gate.to(device))
    check(got, expected * torch.sigmoid(gate.double()).reshape(expected.shape))


def test_rows_out_of_sight_may_hold_anything(device):
    """Values and keys no query sees, or that only later queries see, never reach a query's output."""
    B, T, H, c, N = 2, 5, 4, 64, 70
    g, q, k, v, _ = inputs(B, T, H, c, N, seed=4)
    positions = torch.tensor([[40, 41, 42, 43, 44], [10, 11, 12, 13, 14]])
    expected, _ = formula(q, k, v, causal(positions, N), c ** -0.5)
    for bad in (float("nan"), float("inf")):
        kd, vd = k.clone(), v.clone()
        kd[0, 45:], vd[0, 45:], kd[1, 15:], vd[1, 15:] = bad, bad, bad, bad
        kd[0, 44], vd[0, 44] = bad, bad  # row 0's last query alone sees this one
        got = kernels.verify_attention(q.to(device), kd.to(device), vd.to(device), positions.to(device), c ** -0.5)
        assert not torch.isfinite(got[0, 4]).any()
        got[0, 4] = expected[0, 4].float().to(device)
        check(got, expected)


@pytest.mark.parametrize("offset", [0, 1])
def test_strides_and_alignment(device, offset):
    """Rows that are not 16-byte aligned run the wave-per-query kernel."""
    B, T, H, c, N = 2, 3, 4, 64, 50
    g, q, k, v, positions = inputs(B, T, H, c, N, seed=5)
    wide = torch.zeros(B, N, 2 * c + 3 + offset, device=device)
    wide[..., offset:offset + c], wide[..., offset + c:offset + 2 * c] = k.to(device), v.to(device)
    expected, _ = formula(q, k, v, causal(positions, N), c ** -0.5)
    check(kernels.verify_attention(q.to(device), wide[..., offset:offset + c], wide[..., offset + c:offset + 2 * c],
                                   positions.to(device), c ** -0.5), expected)


def test_a_caller_without_a_workspace_and_the_static_entry(device):
    B, T, H, c, N = 2, 5, 4, 64, 400
    g, q, k, v, positions = inputs(B, T, H, c, N, seed=6)
    expected, _ = formula(q, k, v, causal(positions, N), c ** -0.5)
    qd, kd, vd, pd = (x.to(device).contiguous() for x in (q, k, v, positions))
    check(kernels.verify_attention(qd, kd, vd, pd, c ** -0.5, static_scratch=True, splits=500), expected)
    out = torch.empty_like(qd)
    for splits in (0, 7, 5000):
        out.zero_()
        _lib.check(_lib.lib().wptv_verify_attention(
            _lib.ptr(qd), _lib.ptr(kd), kd.stride(0), kd.stride(1), _lib.ptr(vd), vd.stride(0), vd.stride(1),
            _lib.dtype_code(qd.dtype), _lib.ptr(pd), 0, None, None, None, B, T, H, c, N, ctypes.c_float(c ** -0.5),
            splits, 0, _lib.ptr(out), None, None, 0, _lib.stream(qd.device)), "verify_attention")
        check(out, expected)


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("c", [64, 128])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_values_out_of_sight_in_every_form(device, c, splits, bad):
    """The visible rows of a tile alone, at both widths' column layouts and in parts: a row that only the last
    query of batch row 0 sees, and rows nobody sees, hold no number."""
    B, T, H, N = 2, 5, 4, 200
    g, q, k, v, _ = inputs(B, T, H, c, N, seed=7)
    positions = torch.tensor([[150, 151, 152, 153, 154], [10, 11, 12, 13, 14]])
    expected, _ = formula(q, k, v, causal(positions, N), c ** -0.5)
    vd = v.clone()
    vd[0, 154:], vd[1, 15:] = bad, bad
    got = kernels.verify_attention(q.to(device), k.to(device), vd.to(device), positions.to(device), c ** -0.5,
                                   splits=splits)
    assert not torch.isfinite(got[0, 4]).any()
    got[0, 4] = expected[0, 4].float().to(device)
    check(got, expected)


@pytest.mark.parametrize("splits", [0, 1, 2])
@pytest.mark.parametrize("c", [64, 128])
def test_a_tree_branch_never_reads_its_siblings_values(device, c, splits):
    """Two branches under one root: the left one's value and key rows hold no number; the right one sees none of it."""
    B, H, prefix = 2, 4, 75
    parents = [-1, 0, 0, 1, 2, 3, 4]  # root; left 1 3 5; right 2 4 6
    g, q, k, v, _ = inputs(B, len(parents), H, c, prefix + len(parents), seed=8)
    seen = torch.zeros(len(parents), prefix + len(parents), dtype=torch.bool)
    seen[:, :prefix] = True
    for i, parent in enumerate(parents):
        if parent >= 0:
            seen[i, prefix:] = seen[parent, prefix:]
        seen[i, prefix + i] = True
    expected, _ = formula(q, k, v, seen.expand(B, -1, -1), c ** -0.5)
    kd, vd = k.clone(), v.clone()
    for i in (1, 3, 5):
        kd[:, prefix + i], vd[:, prefix + i] = float("nan"), float("nan")
    base = torch.full((B,), prefix, device=device)
    masks = kernels.tree_ancestors(parents).to(device)
    got = kernels.verify_attention(q.to(device), kd.to(device), vd.to(device), None, c ** -0.5, tree=(base, masks),
                                   splits=splits)
    assert not torch.isfinite(got[:, [1, 3, 5]]).any()
    got[:, [1, 3, 5]] = expected[:, [1, 3, 5]].float().to(device)
    check(got, expected)


@pytest.mark.parametrize("c", [64, 128])
def test_a_ring_slot_outside_the_window_may_hold_anything(device, c):
    """Slots of tokens before the window of every query, and between two queries' windows, hold no number."""
    B, T, H, window, past = 2, 3, 4, 32, 300
    g, q, k, v, positions = inputs(B, T, H, c, past + T, seed=9)
    sink = torch.randn(H, generator=g)
    expected, _ = formula(q, k, v, causal(positions, past + T, window), c ** -0.5, sink)
    ring = torch.full((B, 64, 2 * c), float("nan"))
    held = torch.arange(past - window + 1, past + T)
    ring[:, held % 64] = torch.cat([k, v], -1)[:, held]
    ring[:, (past - window + 1) % 64, c:] = float("inf")  # the first query's first row, the others' none
    got = kernels.ring_attention(q.to(device), ring.to(device), positions.to(device), c ** -0.5, window,
                                 sink.to(device))
    assert not torch.isfinite(got[:, 0]).any()
    got[:, 0] = expected[:, 0].float().to(device)
    check(got, expected)


def test_one_part_gives_a_query_the_same_bits_in_any_batch_and_table(device):
    """The library's own part count follows the batch and the table's length, and the sums' order with it."""
    B, T, H, c, N = 6, 5, 4, 64, 500
    g, q, k, v, positions = inputs(B, T, H, c, N, seed=10)
    table = torch.cat([k, v], -1).to(device)
    qd, pd = q.to(device), positions.to(device)
    whole = kernels.verify_attention(qd, table[..., :c], table[..., c:], pd, c ** -0.5, splits=1)
    longer = torch.cat([table, torch.zeros(B, 700, 2 * c, device=device)], 1)
    for b in range(B):
        for t in (table, longer):
            one = t[b:b + 1]
            alone = kernels.verify_attention(qd[b:b + 1], one[..., :c], one[..., c:], pd[b:b + 1], c ** -0.5, splits=1)
            assert torch.equal(alone[0], whole[b])
