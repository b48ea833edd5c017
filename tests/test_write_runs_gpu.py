"""GPU tests of the cache writes where the runs of consecutive slots start anywhere.

The write kernel stores 16 tokens that fill one aligned 16-slot cell together,
wherever they sit among the input tokens, and the rest one by one, in two
launch forms (few and many rows).  These cases put cell starts at every
position of a 16-token window, end sequences on both sides of cell edges,
break runs with skipped slots and swapped tokens, and cross the row count at
which the form changes.  Every byte of the caches and scales must equal the
oracle's, the untouched slots included.
"""

import numpy as np
import pytest
import torch

from oracle import paged_decode_ref as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def _lib(built):
    import pa_int8

    pa_int8.ext()


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def ragged_slots(tokens, bs, rng, breaks):
    """Slots of `tokens` tokens: sequences of 1..70 tokens that start anywhere in
    their first block; with `breaks`, also skipped tokens, swapped neighbours and
    tokens past the pool.  Returns (slots, blocks of the pool)."""
    parts, used, nb = [], 0, 0
    while used < tokens:
        n = int(min(tokens - used, rng.integers(1, 71)))
        first = int(rng.integers(0, 2) * rng.integers(0, bs))
        blocks = (first + n + bs - 1) // bs
        parts.append(nb * bs + first + np.arange(n))
        nb += blocks
        used += n
    slots = np.concatenate(parts).astype(np.int64)
    perm = rng.permutation(nb)
    slots = perm[slots // bs] * bs + slots % bs
    if breaks:
        # (disjoint pairs: no slot may appear twice)
        i = 2 * rng.choice(tokens // 2, size=max(1, tokens // 60), replace=False)
        slots[i], slots[i + 1] = slots[i + 1].copy(), slots[i].copy()
        slots[rng.random(tokens) < 0.02] = -1
        slots[rng.random(tokens) < 0.005] = nb * bs + 3
    return slots, nb


# (tokens, kv heads): one window, window edges, the last tokens of the few-rows
# form and the first of the many-rows form (4096 waves, four per window and head)
SIZES = [(1, 1), (15, 2), (16, 1), (17, 2), (31, 1), (33, 8), (250, 2), (8191, 2), (8193, 2),
         (16384 + 5, 1)]


@pytest.mark.parametrize("breaks", [False, True])
@pytest.mark.parametrize("mode", ["int8", "fp16"])
@pytest.mark.parametrize("head_dim,block_size", [(128, 16), (72, 32), (256, 128), (8, 64)])
@pytest.mark.parametrize("tokens,hkv", SIZES)
def test_write_runs(tokens, hkv, head_dim, block_size, mode, breaks):
    import pa_int8

    if tokens > 1000 and head_dim == 256:
        tokens, hkv = tokens // 4 + 1, hkv * 4       # the same rows in less memory per token
    rng = np.random.default_rng(tokens * 31 + hkv + head_dim + breaks)
    if breaks and tokens == 1:
        pytest.skip("one token has no run to break")
    slots, nb = ragged_slots(tokens, block_size, rng, breaks)
    k = rng.standard_normal((tokens, hkv, head_dim)).astype(np.float16)
    v = rng.standard_normal((tokens, hkv, head_dim)).astype(np.float16)
    if mode == "fp16":
        kc = rng.standard_normal((nb, hkv, head_dim // 8, block_size, 8)).astype(np.float16)
        vc = rng.standard_normal((nb, hkv, head_dim, block_size)).astype(np.float16)
        tk, tv = _t(kc), _t(vc)
        pa_int8.reshape_and_cache(_t(k), _t(v), tk, tv, _t(slots))
        ok = (slots >= 0) & (slots < nb * block_size)
        blk, off = slots[ok] // block_size, slots[ok] % block_size
        kc[blk, :, :, off] = k[ok].reshape(-1, hkv, head_dim // 8, 8)
        vc[blk, :, :, off] = v[ok]
        got, want = [tk, tv], [kc, vc]
    else:
        kc = rng.integers(-128, 128, size=(nb, hkv, head_dim // 8, block_size, 8)).astype(np.int8)
        vc = rng.integers(-128, 128, size=(nb, hkv, head_dim, block_size)).astype(np.int8)
        ks = rng.standard_normal((nb, hkv, block_size)).astype(np.float32)
        vs = rng.standard_normal((nb, hkv, block_size)).astype(np.float32)
        got = [_t(kc), _t(vc), _t(ks), _t(vs)]
        pa_int8.reshape_and_cache_int8(_t(k), _t(v), *got, _t(slots))
        ref.reshape_and_cache_int8(k, v, slots, kc, vc, ks, vs)
        want = [kc, vc, ks, vs]
    for name, g, w in zip(("k_cache", "v_cache", "k_scales", "v_scales"), got, want):
        g = g.cpu().numpy()
        bad = np.argwhere(g.view(np.uint8).reshape(-1) != w.view(np.uint8).reshape(-1))
        assert bad.size == 0, f"{name}: {len(bad)} bytes differ, first at byte {bad[0][0]}"


# (tokens, kv heads) on both sides of where the few-rows form ends: 2048 waves (fp16, head_dim
# 256), 3072 (fp16; INT8 at 256) and 4096 (INT8), two per window and head; 704, one-wave work-groups
@pytest.mark.parametrize("breaks", [False, True])
@pytest.mark.parametrize("mode", ["int8", "fp16"])
@pytest.mark.parametrize("head_dim,tokens,hkv", [(256, 2048, 8), (256, 2049, 8), (256, 3072, 8),
                                                 (256, 3073, 8), (128, 12288, 2), (128, 12289, 2),
                                                 (128, 16384, 2), (128, 16385, 2), (128, 2816, 2),
                                                 (128, 2817, 2)])
def test_write_runs_at_the_forms_edges(head_dim, tokens, hkv, mode, breaks):
    if tokens > 1000 and head_dim == 256:
        tokens, hkv = 4 * tokens - 4, hkv // 4       # (as test_write_runs maps them back)
    test_write_runs(tokens, hkv, head_dim, 16, mode, breaks)
