"""Radiance cache kernels at the sizes where their splits can go wrong: one
16-row tile, a last wave without a tile, more tiles than resident waves, and
tables whose levels are all hashed, dense and hashed in the same wave step, or
mostly dense."""
from __future__ import annotations

import numpy as np
import pytest

from doonengine_amd import scenes
from doonengine_amd._hip import DeviceBuffer
from doonengine_amd.volume import RadianceCache, Volume, rc_pack_weights, rc_unpack_weights
from oracle import radiance_cache as orc

pytestmark = pytest.mark.gpu

EXTENT = 128.0


@pytest.fixture(scope="module")
def volume(gpu):
    sc = scenes.config_small()
    with Volume(sc.map_size, min_chunks=64) as vol:
        yield vol


def make_rows(rng, n):
    s = np.zeros((n, 16), np.float32)
    s[:, 0:3] = rng.uniform(-2.0, EXTENT + 2.0, (n, 3))        # past the extent on both sides
    s[0, 0:3] = (0.0, EXTENT, 0.5 * EXTENT)
    nrm = rng.normal(size=(n, 3))
    s[:, 3:6] = nrm / np.linalg.norm(nrm, axis=1, keepdims=True)
    s[:, 6:9] = rng.uniform(0.1, 0.9, (n, 3))
    s[:, 9:12] = rng.uniform(0.0, 1.0, (n, 3))
    s[:, 12] = 1.0
    s[:, 13:16] = rng.uniform(0.0, 0.5, (n, 3))
    return s


@pytest.mark.parametrize("log2,n", [(10, 16), (14, 48), (15, 1040), (17, 4096 + 16), (19, 49152 + 80)])
def test_a_batch_predicts_what_its_tiles_do(volume, log2, n):
    """A row's prediction does not depend on the batch it comes in: 16-row calls
    (whose outputs the oracle test checks) give the batch's bits."""
    rng = np.random.default_rng(log2 * 1000 + n)
    cfg = orc.Config(log2_table=log2, extent=EXTENT)
    mats, table = orc.init_params(cfg, seed=9)
    table = rng.normal(0, 0.1, table.shape).astype(np.float32)
    rows = make_rows(rng, n)
    rc = RadianceCache(volume, log2Table=log2, extent=EXTENT, samplesPerFrame=16)
    try:
        rc.set_params(rc_pack_weights(mats), table.reshape(-1))
        out, one = DeviceBuffer(n * 16), DeviceBuffer(16 * 16)
        rc.predict_samples(DeviceBuffer.from_array(rows), n, out)
        volume.synchronize()
        y = out.download(np.float32, (n, 4))
        assert np.all(y[:, 3] == 1.0) and np.all(np.isfinite(y)) and np.abs(y[:, :3] - rows[:, 13:16]).max() > 0.0
        for t in sorted({0, 1 % (n // 16), n // 32, n // 16 - 2 if n > 16 else 0, n // 16 - 1}):
            rc.predict_samples(DeviceBuffer.from_array(rows[16 * t:16 * t + 16]), 16, one)
            volume.synchronize()
            assert np.array_equal(one.download(np.uint32, (16, 4)), y[16 * t:16 * t + 16].view(np.uint32)), t
    finally:
        rc.close()


@pytest.mark.parametrize("log2,n,narrow", [(8, 4096, False), (13, 4112, False), (14, 20000, False), (16, 4096, True),
                                           (8, 12288, False), (13, 12304, False), (16, 16400, True),
                                           (19, 32784, False), (19, 65536, True)])
def test_many_rows_gradients_match_oracle(volume, log2, n, narrow):
    """Table gradients sorted by bucket: tables smaller than a bucket, levels of
    one and of many buckets, and (narrow: all rows within a few cells) buckets of
    several slices. Relative Frobenius error as for the small batches."""
    rng = np.random.default_rng(log2 * 1000 + n)
    cfg = orc.Config(log2_table=log2, extent=EXTENT)
    mats, table = orc.init_params(cfg, seed=3)
    table = rng.normal(0, 0.05, table.shape).astype(np.float32)
    rows = make_rows(rng, n)
    if narrow:
        rows[:, 0:3] = rng.uniform(40.0, 44.0, (n, 3))
    rows[:, 13:16] = 0.0
    rc = RadianceCache(volume, log2Table=log2, extent=EXTENT, samplesPerFrame=16)
    try:
        rc.set_params(rc_pack_weights(mats), table.reshape(-1))
        rc.train_samples(DeviceBuffer.from_array(rows), n, step=False)
        _, _, _, tg = rc.get_params()
        tg = tg.reshape(table.shape).astype(np.float64)
        rc.train_samples(DeviceBuffer.from_array(rows), n, step=False)
        _, _, _, twice = rc.get_params()
    finally:
        rc.close()
    pos = np.clip(rows[:, 0:3], 0.0, EXTENT)
    ref = orc.forward_backward(cfg, mats, table, pos, rows[:, 3:6], rows[:, 6:9], rows[:, 9:12], bf16_ops=True)
    d = ref["dtable"]
    assert np.linalg.norm(tg - d) / np.linalg.norm(d) < 5e-3
    assert np.linalg.norm(twice.reshape(table.shape) - 2.0 * tg) / np.linalg.norm(tg) < 1e-5      # calls add up


@pytest.mark.parametrize("n", [16, 112, 128, 144, 2048 + 16, 32768 + 48])
def test_weight_gradients_at_block_edges(volume, n):
    """Weight gradients are multiplied per block of eight 16-row tiles: one tile, one
    short of a block, a block, one more, and more blocks than the grid has. Rows
    without weight (valid 0) among them."""
    rng = np.random.default_rng(n)
    cfg = orc.Config(log2_table=12, extent=EXTENT)
    mats, table = orc.init_params(cfg, seed=4)
    table = rng.normal(0, 0.05, table.shape).astype(np.float32)
    rows = make_rows(rng, n)
    rows[:, 13:16] = 0.0
    rc = RadianceCache(volume, log2Table=12, extent=EXTENT, samplesPerFrame=16)
    try:
        rc.set_params(rc_pack_weights(mats), table.reshape(-1))
        rc.train_samples(DeviceBuffer.from_array(rows), n, step=False)
        g = rc_unpack_weights(rc.get_params()[2])
        rows[:, 12] = 0.0
        rc.train_samples(DeviceBuffer.from_array(rows), n, step=False)
        again = rc_unpack_weights(rc.get_params()[2])
    finally:
        rc.close()
    pos = np.clip(rows[:, 0:3], 0.0, EXTENT)
    ref = orc.forward_backward(cfg, mats, table, pos, rows[:, 3:6], rows[:, 6:9], rows[:, 9:12], bf16_ops=True)
    for i, (a, b, c) in enumerate(zip(g, ref["dW"], again)):
        assert np.linalg.norm(a - b) / np.linalg.norm(b) < 5e-3, i
        assert np.array_equal(a, c), i
