"""GPU parity of the HSDR encoder (csdr_hsdr_encode, csdr_hsdr_compress) through the C-ABI.

Bars:
  * matching pursuit: codes bit-exact against the reference's compress fixtures (given the
    stream's dictionary) and against the oracle (pinned in test_hsdr_encode_oracle.py) on
    larger random cases; K, tile sizes with and without an 8-element chunk, many tiles per
    workgroup and one;
  * compress, with and without K-SVD passes: the reference's stream byte for byte, on any
    host CPU (the initialisation takes the approximate reciprocal square root of the CPU the
    fixtures were written on from a table, and sums the tile norms in the reference build's
    order; the fixtures were written with one OpenMP thread).
"""
import os

import numpy as np
import pytest

import oracle
from test_hsdr_encode_oracle import stream_parts, tiles_of

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(__file__), "golden")


@pytest.fixture(scope="module")
def enc():
    return np.load(os.path.join(GOLDEN, "hsdr_encode_fixtures.npz"), allow_pickle=False)


def n_cases(enc):
    return len([k for k in enc.files if k.startswith("enc_") and k.endswith("_stream")])


def gpu_codes(gpu, tiles, D, g, S, k):
    from cortexsdr_amd import encode

    t = gpu.from_numpy(np.array(tiles, np.float32)).cuda()
    d = gpu.from_numpy(np.array(D, np.float32)).cuda()
    return encode.encode(t, d, g, S, k).cpu().numpy().view(np.uint16)


def test_encode_matches_reference_fixtures(gpu, enc):
    for i in range(n_cases(enc)):
        v, D, g, codes = stream_parts(enc[f"enc_{i}_stream"].tobytes())
        t = tiles_of(enc[f"enc_{i}_w"], v.tile_rows, v.tile_cols)
        got = gpu_codes(gpu, t, D, g, v.n_stages, v.k_per_stage)
        assert np.array_equal(got, codes), f"case {i}"


@pytest.mark.parametrize("n,C,K,S,k", [(1000, 64, 256, 3, 5), (333, 200, 100, 2, 8),
                                       (40, 1024, 512, 3, 4), (7, 4096, 64, 2, 3),
                                       (1, 8, 8, 2, 4), (500, 60, 64, 2, 3), (300, 39, 48, 3, 2),
                                       (64, 5, 8, 2, 2), (2000, 100, 128, 2, 4)])
def test_encode_matches_oracle(gpu, n, C, K, S, k):
    rng = np.random.default_rng(n + C + K)
    t = (rng.standard_normal((n, C)) * 0.02).astype(np.float32)
    D = rng.standard_normal((K, C)).astype(np.float32)
    D /= np.linalg.norm(D, axis=1, keepdims=True)
    D *= 0.02 * np.sqrt(C / (S * k))
    g = (0.5 ** np.arange(S)).astype(np.float32)
    want = oracle.hsdr_mp(t, D, g, S, k)
    got = gpu_codes(gpu, t, D, g, S, k)
    assert np.array_equal(got, want)


# Each tiles-per-workgroup instantiation of the matching-pursuit kernel (1: the large-tile LDS
# fallback; 4 and 8: what matrices of >= 4096 tiles take, with 2 atoms per lane group and
# float4 tile loads), forced through the kernel's selection override, bit-exact against the
# oracle; ragged last workgroups (n not a multiple of TT), tiles with an 8-element chunk
# (C % 16 == 8) and without, and a case whose natural selection is TT = 1 (C x K too large
# for two tiles under the soft LDS size).
@pytest.mark.parametrize("tt", [1, 4, 8])
@pytest.mark.parametrize("n,C,K,S,k", [(203, 72, 128, 3, 4), (1031, 64, 256, 3, 5),
                                       (37, 200, 64, 2, 8), (45, 896, 160, 3, 3)])
def test_encode_tiles_per_workgroup_match_oracle(gpu, monkeypatch, tt, n, C, K, S, k):
    monkeypatch.setenv("CSDR_HSDR_TILES_PER_WG", str(tt))
    rng = np.random.default_rng(7 * n + C + K + tt)
    t = (rng.standard_normal((n, C)) * 0.02).astype(np.float32)
    D = rng.standard_normal((K, C)).astype(np.float32)
    D /= np.linalg.norm(D, axis=1, keepdims=True)
    D *= 0.02 * np.sqrt(C / (S * k))
    g = (0.5 ** np.arange(S)).astype(np.float32)
    want = oracle.hsdr_mp(t, D, g, S, k)
    got = gpu_codes(gpu, t, D, g, S, k)
    assert np.array_equal(got, want), f"TT={tt}"


# The Gram-matrix form of matching pursuit against the oracle where its bound has to give way:
# atoms held twice (exact ties), zero tiles, tiles far outside the bounded range, zero atoms,
# K off the wave's multiples and each scores-per-lane size, unaligned tile lengths.
@pytest.mark.parametrize("n,C,K,S,k", [(200, 64, 65, 3, 4), (130, 39, 256, 2, 5),
                                       (150, 100, 300, 2, 4), (90, 200, 520, 2, 3),
                                       (70, 33, 1030, 1, 5), (65, 8, 8, 2, 8)])
def test_encode_ties_and_odd_tiles_match_oracle(gpu, monkeypatch, n, C, K, S, k):
    monkeypatch.delenv("CSDR_HSDR_TILES_PER_WG", raising=False)
    rng = np.random.default_rng(n + C + K)
    t = (rng.standard_normal((n, C)) * 0.02).astype(np.float32)
    t[3] = 0
    t[5] *= np.float32(1e-20)
    t[6] *= np.float32(1e15)
    t[8] = t[9]
    D = t[rng.integers(16, n, K)].copy()   # duplicates, and atoms that are tiles
    D /= np.linalg.norm(D, axis=1, keepdims=True)
    D *= 0.02 * np.sqrt(C / (S * k))
    D[K // 2] = 0
    D = D.astype(np.float32)
    g = (0.5 ** np.arange(S)).astype(np.float32)
    assert np.array_equal(gpu_codes(gpu, t, D, g, S, k), oracle.hsdr_mp(t, D, g, S, k))


# Tiles left to projections, by the hundred and the thousand: in the first chunk of tiles (2^24 / K)
# either side of the 256 that go one a workgroup, a count off the tiles per workgroup (4 at K =
# 2048, 8 at K = 64), and in a second chunk, whose tiles and codes are at an offset, a few.
@pytest.mark.parametrize("n,C,K,S,k,n_left", [(8192 + 300, 8, 2048, 2, 2, 1201),
                                              (9001, 24, 64, 2, 3, 9001),
                                              (8192 + 9, 8, 2048, 1, 3, 256),
                                              (5000, 20, 64, 2, 2, 257)])
def test_encode_many_tiles_left_match_oracle(gpu, monkeypatch, n, C, K, S, k, n_left):
    monkeypatch.delenv("CSDR_HSDR_TILES_PER_WG", raising=False)
    rng = np.random.default_rng(n + K)
    t = (rng.standard_normal((n, C)) * 0.02).astype(np.float32)
    D = rng.standard_normal((K, C)).astype(np.float32)
    D *= 0.02 * np.sqrt(C / (S * k)) / np.linalg.norm(D, axis=1, keepdims=True)
    left = rng.permutation(min(n, 8192) if n_left < n else n)[:n_left]
    t[left] *= np.where(rng.random((n_left, 1)) < 0.5, 1e-15, 1e15).astype(np.float32)
    if n_left < n:
        t[8192 + 2:8192 + 60:3] *= np.float32(1e15)
    g = (0.5 ** np.arange(S)).astype(np.float32)
    assert np.array_equal(gpu_codes(gpu, t, D, g, S, k), oracle.hsdr_mp(t, D, g, S, k))


@pytest.mark.parametrize("zero_atom,scale", [(True, 1.0), (False, 1.0), (True, np.inf)])
def test_encode_zero_tiles_match_oracle(gpu, monkeypatch, zero_atom, scale):
    """Zero tiles where atom 0, their first pick, is all zeros (it then stands at every pick), and
    where it is not, its values as small as fp32 holds included; and with an infinite stage
    scale, which makes NaN of the zeros."""
    monkeypatch.delenv("CSDR_HSDR_TILES_PER_WG", raising=False)
    n, C, K, S, k = 300, 100, 200, 3, 4
    rng = np.random.default_rng(5)
    t = (rng.standard_normal((n, C)) * 0.02).astype(np.float32)
    t[::2] = 0
    t[4, 60] = -0.0
    D = (rng.standard_normal((K, C)) * 0.01).astype(np.float32)
    D[0] = 0
    D[9:40] = 0
    D[12, 99] = 1e-38
    if not zero_atom:
        D[0, 70] = 1e-30
    g = (scale * 0.5 ** np.arange(S)).astype(np.float32)
    want = oracle.hsdr_mp(t, D, g, S, k)
    assert (zero_atom and scale == 1.0) == (not want.reshape(n, -1)[::2].any())
    assert np.array_equal(gpu_codes(gpu, t, D, g, S, k), want)


def test_encode_more_picks_than_the_gram_form_holds(gpu, monkeypatch):
    # 32 x 345 picks and their gains are past 64 KiB of LDS: mp_kernel, which keeps none
    monkeypatch.delenv("CSDR_HSDR_TILES_PER_WG", raising=False)
    rng = np.random.default_rng(32)
    t = (rng.standard_normal((4, 8)) * 0.02).astype(np.float32)
    D = (rng.standard_normal((512, 8)) * 0.01).astype(np.float32)
    g = (0.5 ** np.arange(32)).astype(np.float32)
    assert np.array_equal(gpu_codes(gpu, t, D, g, 32, 345), oracle.hsdr_mp(t, D, g, 32, 345))


def test_encode_large_tile_falls_back_to_one_per_workgroup(gpu, monkeypatch):
    # 2 x (C + K) x 4 bytes > 64 KiB: the natural choice is one tile per workgroup
    monkeypatch.delenv("CSDR_HSDR_TILES_PER_WG", raising=False)
    n, C, K, S, k = 9, 4096, 4096, 2, 3
    rng = np.random.default_rng(11)
    t = (rng.standard_normal((n, C)) * 0.02).astype(np.float32)
    D = rng.standard_normal((K, C)).astype(np.float32)
    D /= np.linalg.norm(D, axis=1, keepdims=True)
    D *= 0.02 * np.sqrt(C / (S * k))
    g = (0.5 ** np.arange(S)).astype(np.float32)
    assert np.array_equal(gpu_codes(gpu, t, D, g, S, k), oracle.hsdr_mp(t, D, g, S, k))


def test_compress_matches_reference(gpu, enc):
    """The whole stream (header, dictionary, stage scales, codes, edge strips) is the
    reference's byte for byte, whatever CPU this host has."""
    from cortexsdr_amd import encode

    for i in range(n_cases(enc)):
        w, ref = enc[f"enc_{i}_w"], enc[f"enc_{i}_stream"].tobytes()
        tr, tc, K, S, k = (int(x) for x in enc[f"enc_{i}_cfg"])
        s = encode.compress(w, tr, tc, K, S, k, ksvd_iters=0, stage_decay=0.5)
        assert len(s) == len(ref)
        v, D, g, codes = stream_parts(s)
        rv, rD, rg, rcodes = stream_parts(ref)
        ulp = np.abs(D.view(np.int32).astype(np.int64) - rD.view(np.int32).astype(np.int64))
        assert ulp.max() == 0, f"case {i}: dictionary differs by {ulp.max()} ulp"
        assert np.array_equal(codes, rcodes), f"case {i}"
        assert s == ref, f"case {i}"
        assert oracle.hsdr_decompress(s).shape == w.shape


def test_compress_refined_matches_reference(gpu, enc):
    """ksvd_iters > 0 (atomUpdateStep then matching pursuit again, per pass): the reference's
    stream byte for byte on any host CPU. Its per-atom corrections are double sums in its user
    order; its tile-norm mean and re-seed norms are sums in the order its -O3 -ffast-math
    AVX2 build executes (the mean with one OpenMP thread, as the fixtures were written); the
    initial dictionary takes the fixtures' CPU's reciprocal square root. Also: the GPU's
    matching pursuit over the reference's own refined dictionary gives its codes."""
    from cortexsdr_amd import encode

    n = len([k for k in enc.files if k.startswith("fit_") and k.endswith("_stream")])
    assert n >= 4
    for i in range(n):
        w, ref = enc[f"fit_{i}_w"], enc[f"fit_{i}_stream"].tobytes()
        tr, tc, K, S, k, it = (int(x) for x in enc[f"fit_{i}_cfg"])
        s = encode.compress(w, tr, tc, K, S, k, ksvd_iters=it, stage_decay=0.5)
        v, D, g, codes = stream_parts(s)
        rv, rD, rg, rcodes = stream_parts(ref)
        ulp = np.abs(D.view(np.int32).astype(np.int64) - rD.view(np.int32).astype(np.int64))
        print(f"fit {i}: dictionary {ulp.max()} ulp, codes {np.mean(codes == rcodes):.5f}")
        assert ulp.max() == 0, f"case {i}"
        assert np.array_equal(codes, rcodes), f"case {i}"
        assert s == ref, f"case {i}"
        t = tiles_of(w, rv.tile_rows, rv.tile_cols)
        assert np.array_equal(gpu_codes(gpu, t, rD, rg, S, k), rcodes), f"case {i}"


# One refinement pass from the initial dictionary and codes, against its sums in numpy. The
# device's residuals hold sqrt(S k) 2^-24 of a tile's norm in fp32 roundings, an atom's share of
# which its users' mean takes to under 2e-6 of its length. Users of few atoms, more than a thread keeps from
# one walk over the codes; code counts off the 8-code pieces; runs past one round of 64 codes;
# tile lengths either side of 64 and 256, where 16, 64 or 256 threads take a tile's residual.
@pytest.mark.parametrize("n,C,K,S,k", [(1003, 24, 3, 2, 3), (3001, 40, 40, 2, 5),
                                       (2800, 16, 64, 3, 8), (61, 24, 5, 1, 5),
                                       (1501, 64, 20, 2, 4), (1103, 65, 20, 2, 4),
                                       (899, 256, 12, 2, 3), (902, 257, 12, 2, 3)])
def test_one_refinement_pass(gpu, n, C, K, S, k):
    from cortexsdr_amd import encode

    w = (np.random.default_rng(n).standard_normal((n, C)) * 0.02).astype(np.float32)
    _, D0, g, c0 = stream_parts(encode.compress(w, 1, C, K, S, k, ksvd_iters=0))
    _, D1, _, c1 = stream_parts(encode.compress(w, 1, C, K, S, k, ksvd_iters=1))
    c0 = c0.reshape(n, S * k)
    idx, coef = c0 & 0x7FFF, np.where(c0 & 0x8000, -1.0, 1.0) * np.repeat(g, k)
    assert len(np.unique(idx)) == K  # no atom is re-seeded
    res = w.astype(np.float64)
    for j in range(S * k):
        res -= coef[:, j:j + 1] * D0[idx[:, j]].astype(np.float64)
    target = np.linalg.norm(w.astype(np.float64), axis=1).mean() / np.sqrt(S * k)
    for a in range(K):
        tile, slot = np.nonzero(idx == a)
        cf = coef[tile, slot]
        new = D0[a] + 0.5 * (cf[:, None] * res[tile]).sum(0) / (cf * cf).sum()
        if np.linalg.norm(new) > 1.5 * target:
            new *= target / np.linalg.norm(new)
        assert np.linalg.norm(D1[a] - new) <= 2e-6 * np.linalg.norm(new), f"atom {a}"
    assert np.array_equal(c1.reshape(n, -1), oracle.hsdr_mp(w, D1, g, S, k).reshape(n, -1))


def test_compress_rejects(gpu):
    from cortexsdr_amd import _lib, encode

    w = np.zeros((10, 64), np.float32)
    with pytest.raises(ValueError):   # fewer tiles than atoms
        encode.compress(w, 1, 64, 16, 2, 2)
    with pytest.raises(_lib.CsdrError):   # K-SVD passes over tiles of more than 32768 values
        encode.compress(np.ones((2, 40000), np.float32), 1, 40000, 1, 1, 1, ksvd_iters=1)
