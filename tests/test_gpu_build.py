"""The index build's k-means iteration and cluster sums: several tiles per wave, results that depend
neither on the call nor on the batch, values of any size and values that are not finite."""
import math

import numpy as np
import pytest
import torch

from oracle import oracle as O
from openattention_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _lists(R, T, C):
    return (torch.empty(R, T, device=DEV, dtype=torch.int32), torch.empty(R, C, device=DEV, dtype=torch.int32),
            torch.empty(R, C, device=DEV, dtype=torch.int32))


def _ids(R, T):
    return (torch.full((R, T), -1, device=DEV, dtype=torch.int32),
            torch.zeros(R, -(-T // 64) * 64, device=DEV, dtype=torch.uint8))


def _two_calls(zraw, cm, T, init, cent0):
    """(ids, centroids) by the assignment and the position-order update."""
    asg, asg8 = _ids(cent0.shape[0], T)
    cent = cent0.clone()
    ops.kmeans_assign(zraw, cm, T, cent, asg, asg8)
    ops.kmeans_update(zraw, cm, T, asg8, init, cent, *_lists(cent0.shape[0], T, cent0.shape[1]))
    return asg, cent


@pytest.mark.parametrize("R,T,C", [(96, 8200, 5), (512, 2113, 64), (260, 4161, 33), (1024, 4097, 17), (1024, 4097, 256)])
def test_kmeans_step_of_several_tiles_per_wave(R, T, C):
    """A Lloyd iteration where a wave takes one, two, four and eight tiles, the last tile, wave and
    segment ragged: ids and centroids against the assignment and the position-order update, and a few
    rows against the restatement.  Whole numbers, so that every dot product is exact; in odd rows the
    tokens change from tile to tile between near the centroids (best distances positive) and far on
    their other side (all negative), in every fifth row also within a tile."""
    print(f"[case] k-means step tiles R={R} T={T} C={C}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(R + T + C)
    z = torch.randint(-3, 4, (R, T, 16), device=DEV, generator=g)
    cent = torch.randint(-3, 4, (R, C, 16), device=DEV, generator=g)
    near = z.abs() + 1
    t = torch.arange(T, device=DEV)
    side = torch.where((t // 64) % 2 == 0, 1, -1)
    z[1::2] = near[1::2] * side[:, None]
    cent[1::2] = cent[1::2].abs() + 1
    z[::5] = near[::5] * torch.where((t // 16) % 3 == 0, 1, -1)[:, None]
    cent[::5] = cent[::5].abs() + 1
    zraw = z.to(torch.bfloat16)
    cm = torch.zeros(R, 16, device=DEV)
    init = torch.randint(0, T, (C,), device=DEV, generator=g, dtype=torch.int32)
    cent0 = cent.float().contiguous()
    asg, ref = _two_calls(zraw, cm, T, init, cent0)
    a, a8 = _ids(R, T)
    got = cent0.clone()
    ops.kmeans_step(zraw, cm, T, init, got, a, a8)
    assert torch.equal(a, asg) and torch.equal(got, ref) and torch.equal(a8[:, :T].int(), a)
    rows = [0, 1, 5, R // 2, R - 2, R - 1]
    want = O.kmeans_assign(z[rows].float().cpu().numpy(), cent0[rows].cpu().numpy())
    assert np.array_equal(a[rows].cpu().numpy(), want)
    c_ref, _ = O.kmeans_update(z[rows].float().cpu().numpy(), want, C, init.cpu().numpy())
    assert np.array_equal(got[rows].cpu().numpy(), c_ref)


def _cancelling(T, C, big):
    """(T, 16) tokens, t and t + 128 of every 256 in one cluster: dimension 0 tells the clusters apart,
    dimension 5 holds big in the one and -big in the other, 6 whole multiples of 2^-30 about 2^-22, 7 one
    or the other."""
    g = torch.Generator(device=DEV).manual_seed(T + C)
    t = torch.arange(T, device=DEV)
    ids = torch.randint(0, C, (T // 256 + 1, 1, 128), device=DEV, generator=g).expand(-1, 2, -1).reshape(-1)[:T]
    sign = torch.where(t % 256 < 128, 1.0, -1.0)
    sign[(t % 256 < 128) & (t + 128 >= T)] = 0.0
    z = torch.zeros(T, 16, device=DEV)
    z[:, 0] = 8.0 * (ids - C // 2)
    z[:, 5] = sign * big
    z[:, 6] = (torch.randn(T, device=DEV, generator=g) * 256).round() * 2.0 ** -30
    z[:, 7] = torch.where(t % 4 < 2, sign * big, z[:, 6])
    cent = torch.zeros(C, 16, device=DEV)
    cent[:, 0] = 8.0 * (torch.arange(C, device=DEV) - C // 2)
    return z.to(torch.bfloat16), cent, ids


@pytest.mark.parametrize("T,C", [(4096, 4), (20001, 16), (70000, 2)])
def test_kmeans_step_sums_have_no_order(T, C):
    """Columns whose mean is tiny against their values (+-2^20 in pairs beside 2^-22): the centroids of
    every call, of every row and of every batch (one to eight tiles per wave) are the same bits, and
    those of the exact mean, also with clusters of more than 2^15 members: the values are multiples of
    2^-30, the sums' unit (2^-51 of 2^21)."""
    print(f"[case] k-means sums without order T={T} C={C}", flush=True)
    z, cent, ids = _cancelling(T, C, 2.0 ** 20)
    init = torch.zeros(C, device=DEV, dtype=torch.int32)
    zd, idc = z.double().cpu().numpy(), ids.cpu().numpy()
    want = np.stack([[np.float32(math.fsum(zd[idc == c, j]) / (idc == c).sum()) for j in range(16)] for c in range(C)])
    for R in (1, 3, 8192 * 2 // (T // 64) + 1, 8192 * 8 // (T // 64) + 1):
        zr = z.expand(R, T, 16).contiguous()
        cm = torch.zeros(R, 16, device=DEV)
        for _ in range(2):
            got = cent.expand(R, C, 16).contiguous()
            ops.kmeans_step(zr, cm, T, init, got)
            assert torch.equal(got, got[:1].expand_as(got)), R
            assert np.array_equal(got[0].cpu().numpy(), want), R


@pytest.mark.parametrize("scale", [2.0 ** -126, 2.0 ** -70, 1.0, 2.0 ** 60, 2.0 ** 121])
def test_kmeans_step_of_values_of_any_size(scale):
    """Values from subnormal zP to the end of the fp32 range, over 20 binades: the mean of each cluster
    within 2^-51 of the segment's bound (a power of two at most twice the largest |z| + |colmean|) of
    the exact one, and its rounding to fp32."""
    R, T, C = 3, 3001, 4
    g = torch.Generator(device=DEV).manual_seed(9)
    z, cent, ids = _cancelling(T, C, 64.0)
    z = (z.float() * 2.0 ** -torch.randint(0, 20, (T, 16), device=DEV, generator=g)).to(torch.bfloat16).float()
    z[:, 0] = 8.0 * (ids - C // 2)
    cm = torch.tensor([0.0, 1.0, 3.0, 1e-6, 0.0, 0.3, 1e-7, 2e-7] * 2, device=DEV)
    cm[0] = 0.0
    zs = (z * scale).to(torch.bfloat16)
    zP = (zs.float() - cm * scale)
    got = (cent * min(scale, 2.0 ** 50) if scale >= 2.0 ** -60 else cent).expand(R, C, 16).contiguous()
    init = torch.zeros(C, device=DEV, dtype=torch.int32)
    asg, asg8 = _ids(R, T)
    ops.kmeans_step(zs.expand(R, T, 16).contiguous(), (cm * scale).expand(R, 16).contiguous(), T, init, got, asg, asg8)
    ids = asg[0].cpu().numpy()
    assert torch.equal(asg, asg[:1].expand_as(asg)) and torch.equal(got, got[:1].expand_as(got))
    zd = zP.double().cpu().numpy()
    top = (zs.float().abs().amax(0) + (cm * scale).abs()).double().cpu().numpy()
    for c in range(C):
        m = ids == c
        if not m.any():
            continue
        for j in range(16):
            want = math.fsum(zd[m, j]) / m.sum()
            err = abs(float(got[0, c, j]) - want)
            assert err <= 2.0 ** -51 * 2 * top[j] + 2.0 ** -24 * abs(want) + 2.0 ** -150, (c, j, err, want)


@pytest.mark.parametrize("R", [2, 1100])
def test_kmeans_step_of_values_that_are_not_finite(R):
    """Infinities and NaN in the projection, a column mean that is infinite or NaN and differences past
    the fp32 range: the clusters and dimensions that hold one are the infinity or NaN that the
    position-order sum gives, all others the same bits."""
    T, C = 4200, 7
    g = torch.Generator(device=DEV).manual_seed(R)
    z = torch.randn(R, T, 16, device=DEV, generator=g).to(torch.bfloat16)
    cm = 0.1 * torch.randn(R, 16, device=DEV, generator=g)
    inf, nan = float("inf"), float("nan")
    for t, j, v in ((5, 2, inf), (2100, 2, -inf), (70, 4, nan), (4199, 15, -inf), (2048, 0, inf)):
        z[0, t, j] = v
    cm[1, 3], cm[R - 1, 6], cm[R - 1, 9] = inf, nan, -3e38
    z[R - 1, 77, 9] = 3e38
    init = torch.arange(C, device=DEV, dtype=torch.int32) * 11
    cent0 = (z.index_select(1, init.long()).float() - cm[:, None]).contiguous()
    asg, ref = _two_calls(z, cm, T, init, cent0)
    a, a8 = _ids(R, T)
    got = cent0.clone()
    ops.kmeans_step(z, cm, T, init, got, a, a8)
    assert torch.equal(a, asg)
    assert torch.equal(torch.nan_to_num(got, 7e37, 3.3e38, -3.3e38), torch.nan_to_num(ref, 7e37, 3.3e38, -3.3e38))
    assert not torch.isfinite(ref[0]).all() and not torch.isfinite(ref[R - 1]).all()


@pytest.mark.parametrize("T,G", [(1, 4), (63, 2), (513, 4), (1500, 2), (4099, 4)])
def test_projection_bound_words(T, G):
    """The projection's bound words: each column's largest |bf16(k W)| over its ragged tiles and waves, the
    sign bit where a value is not finite; an iteration with them gives the bits of one without."""
    print(f"[case] bound words T={T} G={G}", flush=True)
    HKV, C = 3, min(T, 6)
    R = HKV * G
    g = torch.Generator(device=DEV).manual_seed(T)
    K = torch.randn(HKV, T, 128, device=DEV, generator=g).to(torch.bfloat16)
    K[1, T - 1, 3] = float("inf")
    W = torch.randn(R, 128, 16, device=DEV, generator=g).to(torch.bfloat16)
    W[2 * G:, :, 5] = 0.0
    zraw = torch.empty(R, T, 16, device=DEV, dtype=torch.bfloat16)
    cm, cm2 = torch.empty(R, 16, device=DEV), torch.empty(R, 16, device=DEV)
    zmax = torch.full((R, 16), -7, device=DEV, dtype=torch.int32)
    ops.qgc_project(K, T, W, G, zraw, cm, zmax=zmax)
    ops.qgc_project(K, T, W, G, torch.empty_like(zraw), cm2)
    assert torch.equal(torch.nan_to_num(cm), torch.nan_to_num(cm2))
    big = zraw.float().abs().amax(1)
    want = torch.where(torch.isfinite(big), big, big.new_tensor(3.3895313892515355e38)).view(torch.int32)
    want = torch.where(torch.isfinite(big), want, want | -(2 ** 31))
    assert torch.equal(zmax, want) and (want[G:2 * G] < 0).all() and (want[2 * G:, 5] == 0).all()
    init = torch.arange(C, device=DEV, dtype=torch.int32)
    cent0 = (zraw.index_select(1, init.long()).float() - cm[:, None]).contiguous()
    a, b = cent0.clone(), cent0.clone()
    ops.kmeans_step(zraw, cm, T, init, a, zmax=zmax)
    ops.kmeans_step(zraw, cm, T, init, b)
    assert torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))


def _cluster_build(K, V, T, asg8, C):
    R = asg8.shape[0]
    nb = torch.empty(R, C, device=DEV)
    S = [torch.full((R, C, 128), 7.0, device=DEV) for _ in range(3)]
    ops.cluster_build(K, V, T, 4, asg8, C, nb, *S, *_lists(R, T, C))
    return nb, S


@pytest.mark.parametrize("T,C", [(255, 1), (256, 1), (4095, 16), (4096, 16), (5001, 5), (700, 9)])
def test_cluster_sums_do_not_depend_on_the_batch(T, C):
    """Cluster statistics of a KV row in a batch of 1, of 3 and of as many as give 16384 (cluster, row)
    pairs, with one and with four waves per cluster (256 mean members up): the same bits, over pairs of
    values about +-2^32 beside values about 2^-12, whose fp64 sums show their order, uneven clusters, an
    empty one, and rows off a 16-byte boundary; within n 2^-53 of the sum of magnitudes of the exact sums,
    and their rounding to fp32."""
    print(f"[case] cluster sums batches T={T} C={C}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(T + C)
    t = torch.arange(T, device=DEV)
    pair = torch.randn(2, 1, T // 2 + 1, 130, device=DEV, generator=g).repeat_interleave(2, 2)[:, :, :T]
    big = pair * torch.where(t % 2 == 0, 2.0 ** 32, -(2.0 ** 32))[:, None]
    one = torch.where((t % 4 < 2)[:, None], big, torch.randn(2, 1, T, 130, device=DEV, generator=g) * 2.0 ** -12)
    one = one.to(torch.bfloat16)
    ids = (C * torch.rand(4, T // 2 + 1, device=DEV, generator=g) ** 2).long().clamp(max=C - 1)
    ids = ids.repeat_interleave(2, 1)[:, :T].clone()
    if C > 3:
        ids[ids == 3] = 4
    base = None
    for B in (1, 3, -(-16384 // (4 * C))):
        if B * T > 1 << 21:
            continue
        kv = one.expand(2, B, T, 130).contiguous()
        asg8 = torch.zeros(4 * B, -(-T // 64) * 64, device=DEV, dtype=torch.uint8)
        asg8[:, :T] = ids.repeat(B, 1)
        nb, S = _cluster_build(kv[0][..., 2:], kv[1][..., 2:], T, asg8, C)
        if base is None:
            base = nb, S
        assert torch.equal(nb, base[0].repeat(B, 1))
        for x, y in zip(S, base[1]):
            assert torch.equal(x, y.repeat(B, 1, 1)), B
    k, v = one[0, 0, :, 2:].double().cpu().numpy(), one[1, 0, :, 2:].double().cpu().numpy()
    for r in (0, 3):
        for c in range(C):
            m = (ids[r] == c).cpu().numpy()
            assert int(base[0][r, c]) == m.sum()
            for got, x in zip(base[1], (k, k * k, v)):
                for j in (0, 77):
                    want = math.fsum(x[m, j])
                    bound = m.sum() * 2.0 ** -53 * np.abs(x[m, j]).sum() + 2.0 ** -24 * abs(want)
                    assert abs(float(got[r, c, j]) - want) <= bound, (r, c, j)


@pytest.mark.parametrize("T,C", [(300, 8), (4097, 16)])
def test_cluster_sums_into_rows_off_16_bytes(T, C):
    """Statistics rows that start 4 bytes off a 16-byte boundary, with one and four waves per cluster: the
    bits of aligned ones."""
    g = torch.Generator(device=DEV).manual_seed(T)
    K, V = (torch.randn(2, T, 128, device=DEV, generator=g).to(torch.bfloat16) for _ in range(2))
    R = 8
    asg8 = torch.zeros(R, -(-T // 64) * 64, device=DEV, dtype=torch.uint8)
    asg8[:, :T] = torch.randint(0, C, (R, T), device=DEV, generator=g)
    nb, S = _cluster_build(K, V, T, asg8, C)
    off = [torch.full((R * C * 128 + 2,), 7.0, device=DEV) for _ in range(3)]
    ops.cluster_build(K, V, T, 4, asg8, C, torch.empty_like(nb), *(t[1:-1].view(R, C, 128) for t in off), *_lists(R, T, C))
    for t, want in zip(off, S):
        assert torch.equal(t[1:-1].view(R, C, 128), want) and t[0] == 7.0 and t[-1] == 7.0
