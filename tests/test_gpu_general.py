"""The general expert-FFN path (MOE355_PATH_SIMT): fp32 layers and sizes the
bf16/f16 tiled kernels do not take, at the edges of its tiles: 16-row tiles up
to ten rows per expert and 64-row tiles above, K steps of 128 and 256 bytes,
feature tiles of 16 to 128, and the 128-row maps that its kernel shares with the
tiled family, against the fp64 oracle (the tolerances of the other paths' tests)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from _helpers import DT, banner, make_bank, skewed_ids
from oracle import oracle
from reframework_amd import _capi
from reframework_amd.moe import fused_experts
from test_gpu_experts import _check, gpu_fused

pytestmark = pytest.mark.gpu

SIMT = _capi.PATH_SIMT


# (H, I): smallest, below one K step, partial last steps and feature tiles of
# either kernel, whole steps of both
SIZES = {"f32": [(4, 4), (20, 36), (132, 68), (64, 128), (260, 324)],
         "bf16": [(8, 8), (24, 40), (136, 200), (320, 72), (264, 520)],
         "f16": [(8, 16), (72, 136), (392, 264)]}


@pytest.mark.parametrize("dts,size", [(d, s) for d, ss in SIZES.items() for s in ss],
                         ids=lambda v: str(v))
@pytest.mark.parametrize("T", [1, 13, 20, 21, 70, 300])
def test_general_path_sizes(dts, size, T, dev):
    H, I = size
    E, K = 4, 2
    dt = DT[dts]
    plan = _capi.make_plan(T, H, I, E, K, _capi.dtype_code(dt))
    assert plan.path == SIMT
    assert plan.tile_rows == (16 if T * K // min(T * K, E) <= 10 else 64)
    banner(f"general {dts} T={T} H={H} I={I} tile={plan.tile_rows} splits={plan.down_splits}")
    w1, w2 = make_bank(E, H, I, dt, seed=H + I)
    x = torch.randn(T, H, generator=torch.Generator().manual_seed(T)).to(dt)
    ids = skewed_ids(T, K, E, seed=T, skew=1.0)
    w = np.random.default_rng(T).random((T, K)).astype(np.float32)
    _check(gpu_fused(x, w1, w2, w, ids), x, w1, w2, w, ids)


@pytest.mark.parametrize("dts,H,I", [("f32", 132, 260), ("bf16", 136, 200)])
@pytest.mark.parametrize("m", [11, 16, 17, 32, 33, 48, 49, 63, 64, 65, 96, 97, 128, 129])
def test_general_path_group_sizes(m, dts, H, I, dev):
    # all m tokens to expert 0 plus one token on expert 3 (expert 1 and 2 empty)
    dt = DT[dts]
    banner(f"general {dts} group of {m}")
    w1, w2 = make_bank(4, H, I, dt, seed=m)
    x = torch.randn(m + 1, H, generator=torch.Generator().manual_seed(m)).to(dt)
    ids = np.zeros((m + 1, 1), np.int64)
    ids[-1, 0] = 3
    w = np.ones((m + 1, 1), np.float32)
    _check(gpu_fused(x, w1, w2, w, ids, path=SIMT), x, w1, w2, w, ids, path=SIMT)


@pytest.mark.parametrize("E,H,I,T,path,tile", [
    # 25 MB of weights: 16-row tiles up to 10 rows per expert
    (4, 640, 1664, 40, _capi.PATH_MFMA_SKINNY, 16), (4, 640, 1664, 44, SIMT, 64),
    (4, 640, 1664, 300, SIMT, 64),
    # 2.4 MB and 7.1 MB: 16-row tiles up to 211 and 70 rows
    (4, 384, 256, 40, _capi.PATH_MFMA_SKINNY, 16), (4, 384, 256, 44, SIMT, 16),
    (4, 384, 256, 847, SIMT, 16), (4, 384, 256, 848, SIMT, 64), (8, 384, 384, 567, SIMT, 16),
    (8, 384, 384, 568, SIMT, 64)])
def test_sizes_only_the_streaming_kernel_tiles(E, H, I, T, path, tile, dev):
    # H a multiple of 128, not of 256
    K = 1
    plan = _capi.make_plan(T, H, I, E, K, _capi.BF16)
    assert (plan.path, plan.tile_rows) == (path, tile)
    banner(f"E={E} H={H} I={I} T={T} path={path}")
    w1, w2 = make_bank(E, H, I, torch.bfloat16, seed=T)
    x = torch.randn(T, H, generator=torch.Generator().manual_seed(T)).to(torch.bfloat16)
    ids = skewed_ids(T, K, E, seed=T, skew=0.5)
    w = np.random.default_rng(T).random((T, K)).astype(np.float32)
    _check(gpu_fused(x, w1, w2, w, ids), x, w1, w2, w, ids)


@pytest.mark.parametrize("m", [31, 33, 96, 97, 128, 129, 191, 193])
@pytest.mark.parametrize("dts,I", [("bf16", 128), ("f16", 640)])
def test_128_row_maps_up_to_64_rows_per_expert(dts, I, m, dev):
    # one large group among three experts: its tile(s) of every 32-row count, y
    # rounded (one K-split) or in fp32 planes; past 64 rows on average the
    # persistent 128-row kernel runs the same plan
    H, E, T = 256, 3, m + 2
    dt = DT[dts]
    plan = _capi.make_plan(T, H, I, E, 1, _capi.dtype_code(dt), _capi.PATH_MFMA_TILED128)
    banner(f"128-row map {dts} I={I} group of {m} splits={plan.down_splits}")
    w1, w2 = make_bank(E, H, I, dt, seed=m)
    x = torch.randn(T, H, generator=torch.Generator().manual_seed(m)).to(dt)
    ids = np.full((T, 1), 1, np.int64)
    ids[0, 0], ids[-1, 0] = 2, 0
    w = np.ones((T, 1), np.float32)
    path = _capi.PATH_MFMA_TILED128
    _check(gpu_fused(x, w1, w2, w, ids, path=path), x, w1, w2, w, ids, path=path)


@pytest.mark.parametrize("E,H,I,T", [(24, 3072, 8192, 480), (24, 3072, 8192, 492),
                                     (16, 4096, 8192, 96)])
def test_128_row_maps_of_more_than_3_gb_of_weights(E, H, I, T, dev):
    """Both sides of that dispatch: the general kernel up to 40 rows per expert,
    the persistent one above and where a matrix is a power of two."""
    K = 2
    banner(f"128-row map E={E} H={H} I={I} T={T}")
    plan = _capi.make_plan(T, H, I, E, K, _capi.BF16)
    assert plan.path == _capi.PATH_MFMA_TILED128 and 6 * E * H * I > 3e9
    g = torch.Generator(device=dev).manual_seed(T)
    w1 = torch.empty(E, 2 * I, H, dtype=torch.bfloat16, device=dev).normal_(0, 0.02, generator=g)
    w2 = torch.empty(E, H, I, dtype=torch.bfloat16, device=dev).normal_(0, 0.02, generator=g)
    x = torch.empty(T, H, dtype=torch.bfloat16, device=dev).normal_(generator=g)
    ids = torch.from_numpy(skewed_ids(T, K, E, seed=T, skew=1.0)).to(dev)
    w = torch.rand(T, K, generator=g, device=dev)
    out = fused_experts(x, w1, w2, w, ids)
    want = torch.zeros(T, H, dtype=torch.float64, device=dev)
    for e in range(E):
        tok, slot = torch.nonzero(ids == e, as_tuple=True)
        gate, up = (x[tok].double() @ w1[e].double().t()).chunk(2, -1)
        y = (gate * torch.sigmoid(gate) * up) @ w2[e].double().t()
        want.index_add_(0, tok, y * w[tok, slot, None].double())
    # bf16 rounds the intermediate, the slot's result and the output once each
    assert (out.double() - want).norm() <= 3 * 2.0 ** -9 * want.norm()
    assert (out.double() - want).abs().max() <= 2e-2 * want.abs().max()


@pytest.mark.parametrize("T", [3, 100])
@pytest.mark.parametrize("dts,H,I", [("f32", 132, 68), ("bf16", 136, 200), ("f16", 256, 128),
                                     ("bf16", 384, 256)])
def test_general_path_element_alignment(dts, H, I, T, dev):
    """Weights and tokens one element off a 16-byte boundary."""
    dt = DT[dts]
    E, K = 4, 2
    banner(f"general {dts} unaligned T={T}")
    w1, w2 = make_bank(E, H, I, dt, seed=1)
    x = torch.randn(T, H, generator=torch.Generator().manual_seed(T)).to(dt)
    ids = skewed_ids(T, K, E, seed=T, skew=0.5)
    w = np.random.default_rng(T).random((T, K)).astype(np.float32)

    def off(t):
        buf = torch.empty(t.numel() + 1, dtype=dt, device=dev)
        buf[1:] = t.reshape(-1).to(dev)
        return buf[1:].view(t.shape)

    d1, d2 = [off(t) for t in w1], [off(t) for t in w2]
    xd, tw, ti = off(x), torch.from_numpy(w).to(dev), torch.from_numpy(ids.astype(np.int32)).to(dev)
    plan = _capi.make_plan(T, H, I, E, K, _capi.dtype_code(dt), SIMT)
    ws = torch.empty(plan.workspace_bytes, dtype=torch.uint8, device=dev)
    out = torch.empty(T, H, dtype=dt, device=dev)
    p1, p2 = [t.data_ptr() for t in d1], [t.data_ptr() for t in d2]
    _capi.permute(plan, ti, ws)
    _capi.gate_up(plan, xd, p1, 0, ws)
    _capi.down(plan, p2, ws)
    _capi.combine(plan, tw, out, False, ws)
    _check(out, x, w1, w2, w, ids, path=SIMT)


@pytest.mark.parametrize("act", [1, 2], ids=["gelu", "gelu_tanh"])
@pytest.mark.parametrize("T", [3, 70])
@pytest.mark.parametrize("dts,H,I", [("f32", 132, 68), ("bf16", 136, 200), ("f16", 256, 144)])
def test_general_path_activations(dts, H, I, T, act, dev):
    E, K = 4, 2
    dt = DT[dts]
    banner(f"general {dts} T={T} activation {act}")
    assert _capi.make_plan(T, H, I, E, K, _capi.dtype_code(dt)).path == SIMT
    w1, w2 = make_bank(E, H, I, dt, seed=act)
    x = torch.randn(T, H, generator=torch.Generator().manual_seed(T)).to(dt)
    ids = skewed_ids(T, K, E, seed=T, skew=0.5)
    w = np.random.default_rng(T).random((T, K)).astype(np.float32)
    _check(gpu_fused(x, w1, w2, w, ids, act=act), x, w1, w2, w, ids, act=act)


@pytest.mark.parametrize("T", [5, 70])
@pytest.mark.parametrize("dts,H,I", [("f32", 132, 68), ("bf16", 136, 200)])
def test_general_path_keeps_infinite_tokens_to_themselves(dts, H, I, T, dev):
    """A token row ends inside a K step and the next one starts with infinities;
    the last one is also what rows past the group read."""
    dt = DT[dts]
    E, K = 2, 1
    banner(f"general {dts} infinite tokens T={T}")
    w1, w2 = make_bank(E, H, I, dt, seed=5)
    ids = np.zeros((T, K), np.int64)
    w = np.ones((T, K), np.float32)
    x = torch.randn(T, H, generator=torch.Generator().manual_seed(T)).to(dt)
    ref = oracle.fused_experts(x, w1, w2, w, ids, activation=0)
    bad = [1, T - 1]
    x[bad, :4] = float("inf")
    got = gpu_fused(x, w1, w2, w, ids).double().cpu().numpy()
    assert not np.isfinite(got[bad]).any()
    keep = np.setdiff1d(np.arange(T), bad)
    assert oracle.max_rel(got[keep], ref[keep]) <= (1e-5 if dt == torch.float32 else 2e-2)


def test_token_rows_past_2_gb(dev):
    """Sizes of the tiled kernels whose tokens exceed their 32-bit offsets run
    the general kernel above 10 rows per expert; tokens from both ends and the
    2 GB boundary against the oracle."""
    T, H, I, E, K = 131100, 8192, 128, 2, 1
    banner(f"token rows past 2 GB T={T} H={H}")
    plan = _capi.make_plan(T, H, I, E, K, _capi.BF16)
    assert T * H * 2 > 1 << 31 and plan.path == SIMT and plan.tile_rows == 64
    w1, w2 = make_bank(E, H, I, torch.bfloat16, seed=8)
    x = torch.empty(T, H, dtype=torch.bfloat16, device=dev).normal_(
        generator=torch.Generator(device=dev).manual_seed(8))
    ids = np.random.default_rng(8).integers(0, E, (T, K))
    w = np.random.default_rng(9).random((T, K)).astype(np.float32)
    out = fused_experts(x, [t.to(dev) for t in w1], [t.to(dev) for t in w2],
                        torch.from_numpy(w).to(dev), torch.from_numpy(ids).to(dev))
    pick = np.r_[0:24, T // 2:T // 2 + 8, 131060:131100]
    _check(out[pick], x[pick].cpu(), w1, w2, w[pick], ids[pick], path=SIMT)


@pytest.mark.parametrize("skew", [1.1, 2.0])
@pytest.mark.parametrize("T,E,K", [(512, 16, 2), (330, 64, 6)])
def test_128_row_maps_with_popular_experts(T, E, K, skew, dev):
    """Full tiles of popular experts beside tiles of a few rows, on 128-row maps
    of at most 64 rows per expert on average."""
    H, I = 256, 384
    plan = _capi.make_plan(T, H, I, E, K, _capi.BF16)
    assert plan.path == _capi.PATH_MFMA_TILED128 and T * K <= 64 * E
    ids = skewed_ids(T, K, E, seed=T, skew=skew)
    assert np.bincount(ids.ravel()).max() > 256
    banner(f"128-row map E={E} T={T} Zipf {skew}")
    w1, w2 = make_bank(E, H, I, torch.bfloat16, seed=T)
    x = torch.randn(T, H, generator=torch.Generator().manual_seed(T)).to(torch.bfloat16)
    w = np.random.default_rng(T).random((T, K)).astype(np.float32)
    _check(gpu_fused(x, w1, w2, w, ids), x, w1, w2, w, ids)


@pytest.mark.parametrize("T", [2, 60])
@pytest.mark.parametrize("dts,H,I", [("f32", 132, 68), ("bf16", 136, 200)])
def test_general_path_keeps_infinities_in_their_row(dts, H, I, T, dev):
    """A weight row ends inside a K step and the next one is infinite: only
    that row's feature is affected."""
    dt = DT[dts]
    E, K, bad = 2, 1, 17
    w1, w2 = make_bank(E, H, I, dt, seed=5)
    ids = np.zeros((T, K), np.int64)
    w = np.ones((T, K), np.float32)
    x = torch.randn(T, H, generator=torch.Generator().manual_seed(T)).to(dt)
    ref = oracle.fused_experts(x, w1, w2, w, ids, activation=0)
    w2[0][bad, 0] = float("inf")
    out = fused_experts(x.to(dev), [t.to(dev) for t in w1], [t.to(dev) for t in w2],
                        torch.from_numpy(w).to(dev), torch.from_numpy(ids).to(dev))
    got = out.float().cpu().numpy().astype(np.float64)
    assert not np.isfinite(got[:, bad]).any()
    keep = np.arange(H) != bad
    assert oracle.max_rel(got[:, keep], ref[:, keep]) <= (1e-5 if dt == torch.float32 else 2e-2)


@pytest.mark.parametrize("T,H,I", [(3, 136, 200), (3, 256, 144), (60, 136, 200)],
                         ids=["streaming general", "streaming plain", "64-row tiles"])
def test_general_path_applies_the_full_precision_activation(T, H, I, dev):
    """SiLU at -88.5 .. -87.5 is about -5e-37: 1 / (1 + e^88) lies below the
    smallest normal fp32 number, which the hardware reciprocal of the other
    families flushes to zero and the fp32 division of this path does not."""
    banner(f"general activation T={T} H={H} I={I}")
    E, dt = 2, torch.bfloat16
    assert _capi.make_plan(T, H, I, E, 1, _capi.BF16).path == SIMT
    g = -87.5 - 0.5 * (torch.arange(I) % 3)              # exact in bf16
    x, w1 = torch.zeros(T, H), torch.zeros(2 * I, H)
    x[:, 0], w1[:I, 0], w1[I:, 0] = 1.0, g, 1.0          # gate g, up 1, both exact
    w2 = torch.zeros(H, I)
    n = min(H, I)
    w2[range(n), range(n)] = 1.0                         # output h is the intermediate h
    ids = np.arange(T)[:, None] % E
    out = gpu_fused(x.to(dt), [w1.to(dt)] * E, [w2.to(dt)] * E, np.ones((T, 1), np.float32), ids)
    want = (g.double() / (1.0 + torch.exp(-g.double())))[:n].numpy()
    got = out.double().cpu().numpy()[:, :n]
    # the intermediate is rounded to bf16 once: 2^-8 of the value, a little for expf
    assert np.max(np.abs(got - want) / np.abs(want)) <= 2.0 ** -8 * 1.01


def test_static_scratch_drops_the_splits(dev):
    """A call whose K-split plan needs more than the static scratch still fits
    it without the splits, as it did before there were any."""
    T, H, I, E, K = 500, 2048, 13056, 2, 2
    plan = _capi.make_plan(T, H, I, E, K, _capi.F32)
    unsplit = plan.off_y + T * K * H * 4
    assert plan.down_splits > 1
    assert unsplit < _capi.STATIC_SCRATCH_BYTES < plan.workspace_bytes
    g = torch.Generator(device=dev).manual_seed(0)
    w1 = torch.empty(E, 2 * I, H, device=dev).normal_(0, 0.02, generator=g)
    w2 = torch.empty(E, H, I, device=dev).normal_(0, 0.02, generator=g)
    x = torch.empty(T, H, device=dev).normal_(generator=g)
    w, ids = torch.topk(torch.softmax(torch.empty(T, E, device=dev).normal_(generator=g), -1), K)
    want = fused_experts(x, w1, w2, w, ids)
    out = torch.empty_like(x)
    _capi.fused_experts_static(x, [w1[e].data_ptr() for e in range(E)],
                               [w2[e].data_ptr() for e in range(E)], I, w.contiguous(),
                               ids.int().contiguous(), 0, out)
    # the same products in fp32, summed in another order
    assert (out - want).norm() <= 1e-5 * want.norm()


def test_more_items_than_one_grid_dimension_holds(dev):
    """2^24 workgroups of 256 threads are past what HIP takes in one grid
    dimension: the general kernel's items go over two."""
    T, H, I = 4096 * 1023, 4, 8448
    plan = _capi.make_plan(T, H, I, 1, 1, _capi.F32)
    assert plan.max_tiles * (I // 32) > 1 << 24
    if torch.cuda.mem_get_info()[0] < plan.workspace_bytes + (4 << 30):
        pytest.skip(f"needs {plan.workspace_bytes >> 30} GiB of GPU memory")
    banner(f"general {plan.max_tiles * (I // 32)} gate_up items")
    w1, w2 = make_bank(1, H, I, torch.float32, seed=3)
    x = torch.randn(4096, H, generator=torch.Generator().manual_seed(3))
    xd, d1, d2 = x.to(dev).repeat(T // 4096, 1), w1[0].to(dev), w2[0].to(dev)
    tw = torch.ones(T, 1, device=dev)
    ids = torch.zeros(T, 1, dtype=torch.int32, device=dev)
    out = torch.full((T, H), float("nan"), device=dev)
    ws = torch.empty(plan.workspace_bytes, dtype=torch.uint8, device=dev)
    _capi.fused_experts(xd, [d1.data_ptr()], [d2.data_ptr()], I, tw, ids, 0, out, ws)
    torch.cuda.synchronize()
    del ws
    torch.cuda.empty_cache()
    # a row's sums do not depend on its place: every repeat is the first one
    assert torch.equal(out.view(-1, 4096 * H), out[:4096].reshape(1, -1).expand(T // 4096, -1))
    ref = oracle.fused_experts(x, w1, w2, np.ones((4096, 1), np.float32),
                               np.zeros((4096, 1), np.int64), activation=0)
    assert oracle.max_rel(out[:4096].double().cpu().numpy(), ref) <= 1e-5
