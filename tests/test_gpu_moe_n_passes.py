"""The batched routed experts' passes (csrc/dsv4_moe_mx.hip, k_mn_prepare and
k_mn_pass) at the sizes where a pass changes shape: an expert with 1 to 12
pairs (each count of term copies per wave, the edge of a column tile, a second
tile, a second pass), both tile forms (experts averaging more than five pairs
take two tiles), unit counts known at compile time and not (hidden 7168 /
inter 2048 against the others), more than 1024 pairs (a larger routing table),
ids that share a table entry, and an infinite activation through the padded
units. Every token's row has the single-token call's bits."""
import ctypes

import numpy as np
import pytest

import common

pytestmark = pytest.mark.gpu


def _experts(gpu, dsv4, layer, ids, hidden, inter, seed):
    rng = np.random.default_rng(seed)
    for e in ids:
        w = common.fp4_expert(rng, hidden, inter)
        ew = dsv4.expert(w["w1"], w["s1"], w["w3"], w["s3"], w["w2"], w["s2"], hidden, inter)
        assert gpu.dsv4_gpu_upload_expert(layer, int(e), ctypes.byref(ew)) == 0
    return rng


def _check(dsv4, layer, X, IDX, W, hidden, inter):
    got = dsv4.moe_fp4_n(X, layer, IDX, W, hidden, inter, 10.0)
    for t in range(X.shape[0]):
        one = dsv4.moe_fp4(X[t], layer, IDX[t], W[t], hidden, inter, 10.0)
        nan = np.isnan(one)
        assert np.array_equal(nan, np.isnan(got[t])), t
        assert common.bits_equal(got[t][~nan], one[~nan]), t


@pytest.mark.parametrize("layer,hidden,inter", [(310, 7168, 2048), (311, 512, 512),
                                                (312, 2560, 1024)])
def test_pairs_per_expert(gpu, dsv4, monkeypatch, layer, hidden, inter):
    """Expert e of 12 is asked for by e + 1 tokens (78 pairs, and 16 experts in
    the layer: at most five each on average, so one tile per pass)."""
    monkeypatch.setenv("DSV4_GPU_MOEN_TOKENWISE", "0")
    rng = _experts(gpu, dsv4, layer, list(range(15)) + [31], hidden, inter, 5)
    pairs = [e for e in range(12) for _ in range(e + 1)]
    IDX = np.array(pairs, np.int32).reshape(39, 2)
    IDX[:, 1] = np.roll(IDX[:, 1], 7)
    X = rng.standard_normal((39, hidden)).astype(np.float32)
    X[3, 5] = np.inf
    W = rng.random((39, 2)).astype(np.float32)
    _check(dsv4, layer, X, IDX, W, hidden, inter)


@pytest.mark.parametrize("layer,nt,topk", [(315, 64, 3), (316, 13, 4), (317, 50, 8)])
def test_two_tiles(gpu, dsv4, monkeypatch, layer, nt, topk):
    """Few experts, so that they average more than five pairs: two column
    tiles per pass, with passes of 1 to 10 pairs."""
    monkeypatch.setenv("DSV4_GPU_MOEN_TOKENWISE", "0")
    hidden, inter = 1024, 512
    rng = _experts(gpu, dsv4, layer, range(8), hidden, inter, 7)
    IDX = np.stack([rng.choice(8, topk, replace=False, p=np.arange(1, 9) / 36.0)
                    for _ in range(nt)]).astype(np.int32)
    X = rng.standard_normal((nt, hidden)).astype(np.float32)
    X[1, 9] = -np.inf
    W = rng.random((nt, topk)).astype(np.float32)
    _check(dsv4, layer, X, IDX, W, hidden, inter)


def test_routing_table_and_colliding_ids(gpu, dsv4, monkeypatch):
    """64 tokens x 32 experts (2048 pairs, a 4096-entry table) over ids that
    are equal modulo every table size."""
    monkeypatch.setenv("DSV4_GPU_MOEN_TOKENWISE", "0")
    hidden, inter, layer = 512, 512, 318
    ids = np.concatenate([np.arange(20), np.arange(20) + 8192]).astype(np.int32)
    rng = _experts(gpu, dsv4, layer, ids, hidden, inter, 9)
    IDX = np.stack([rng.choice(ids, 32, replace=False) for _ in range(64)]).astype(np.int32)
    X = rng.standard_normal((64, hidden)).astype(np.float32)
    W = rng.random((64, 32)).astype(np.float32)
    _check(dsv4, layer, X, IDX, W, hidden, inter)
