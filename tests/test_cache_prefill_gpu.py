"""GPU tests of PagedKVCache.prefill's fused write: the per-tensor scales taken on
the device, and the rest of the last block zeroed by the write itself.

Expected: the scale formula of benchmarks/int8_bridge/paged_cache.py:101-102 on
the CPU, then the per-op write (checked against the oracle elsewhere) into a
second cache and zeros in the tail.  Every byte and scale bit must match.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def _lib(built):
    import pa_int8

    pa_int8.ext()


def tensor_scale(x):
    return (x.cpu().abs().amax() / 127.0).to(torch.float32).clamp_min(1e-8).reshape(1).to(DEV)


def rows(tokens, hkv, d, dtype, strided, seed):
    g = torch.Generator().manual_seed(seed)
    if strided:     # views of a wider row: neither head nor token stride is dense
        t = torch.randn(tokens, hkv + 3, 2 * d, generator=g).to(dtype).to(DEV)
        return t[:, 1:1 + hkv, :d], t[:, 2:2 + hkv, d:]
    return (torch.randn(tokens, hkv, d, generator=g).to(dtype).to(DEV),
            torch.randn(tokens, hkv, d, generator=g).to(dtype).to(DEV))


def bits(t):
    return t.contiguous().view(torch.uint8)


# one token, tails of every length class, several work-groups, the last piece of a
# work-group's share and one past it (8 loads x 512 threads x 8 elements at 2 x 128)
@pytest.mark.parametrize("tokens", [1, 15, 16, 17, 127, 128, 129, 700, 4001])
@pytest.mark.parametrize("variant", ["fp16", "int8_per_token", "int8_per_tensor"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("head_dim,block_size,strided", [(128, 16, False), (72, 64, True),
                                                         (256, 32, False)])
def test_prefill_matches_per_op_write(tokens, variant, dtype, head_dim, block_size, strided):
    import pa_int8

    hkv = 2
    k, v = rows(tokens, hkv, head_dim, dtype, strided, tokens + head_dim)
    cap = tokens + 2 * block_size
    got, want = (pa_int8.PagedKVCache(2, hkv, head_dim, cap, block_size=block_size, variant=variant,
                                      device=DEV) for _ in range(2))
    for c in (got, want):     # an earlier, longer prompt: its tail must go
        for t in c._tensors():
            t.fill_(3)
    got.prefill(1, k, v)
    slots = want._slots[:tokens]
    kc, vc = want.k_cache[1], want.v_cache[1]
    if variant == "fp16":
        pa_int8.reshape_and_cache(k.half(), v.half(), kc, vc, slots)
    elif variant == "int8_per_token":
        pa_int8.reshape_and_cache_int8(k, v, kc, vc, want.k_scales[1], want.v_scales[1], slots)
    else:
        sk, sv = tensor_scale(k), tensor_scale(v)
        assert torch.equal(bits(got._k_tensor_scale[1]), bits(sk))
        assert torch.equal(bits(got._v_tensor_scale[1]), bits(sv))
        pa_int8.reshape_and_cache_int8_static(k, v, kc, vc, want.k_scales[1], want.v_scales[1],
                                              slots, sk, sv)
    off = tokens % block_size
    if off:
        for name, (_, _, axis) in want.layout.tensors().items():
            getattr(want, name)[1, tokens // block_size].narrow(axis, off, block_size - off).zero_()
    for g, w in zip(got._tensors(), want._tensors()):
        assert torch.equal(bits(g), bits(w))
    assert got.lengths == [0, tokens]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("value", [0.0, 1e-7, -65504.0, float("inf"), float("nan"), 3.0])
def test_tensor_scale_special_values(dtype, value):
    """amax of zeros, tiny values, the type's ends, infinity and NaN, placed in the
    last element; three calls in a row leave the shared counter usable."""
    import pa_int8

    k = torch.zeros(33, 2, 64, dtype=dtype, device=DEV)
    v = torch.full_like(k, 0.5)
    k[-1, -1, -1] = value
    c = pa_int8.PagedKVCache(1, 2, 64, 64, variant="int8_per_tensor", device=DEV)
    for _ in range(3):
        c.prefill(0, k, v)
        for got, x in ((c._k_tensor_scale[0], k), (c._v_tensor_scale[0], v)):
            want = tensor_scale(x)
            if torch.isnan(want).any():
                assert torch.isnan(got).all()
            else:
                assert torch.equal(bits(got), bits(want))


def test_every_tensor_scale():
    """The scale of every fp16 and bf16 magnitude equals torch's."""
    import pa_int8

    for dtype in (torch.float16, torch.bfloat16):
        mags = torch.arange(0, 1 << 15, dtype=torch.int32).to(torch.int16).view(dtype).to(DEV)
        c = pa_int8.PagedKVCache(1, 1, 8, 16, variant="int8_per_tensor", device=DEV)
        got = []
        for x in mags.view(-1, 1, 1, 1).expand(-1, 1, 1, 8).contiguous():
            c.prefill(0, x, x)
            got.append(c._k_tensor_scale[0])
        got = torch.cat(got)
        want = (mags.cpu() / 127.0).to(torch.float32).clamp_min(1e-8).to(DEV)
        ok = torch.isnan(want)
        assert torch.equal(torch.isnan(got), ok)
        assert torch.equal(got[~ok], want[~ok])


def test_empty_prompt():
    import pa_int8

    e = torch.zeros(0, 2, 64, dtype=torch.float16, device=DEV)
    c = pa_int8.PagedKVCache(1, 2, 64, 64, variant="int8_per_token", device=DEV)
    c.prefill(0, e, e)
    assert c.lengths == [0]
    c = pa_int8.PagedKVCache(1, 2, 64, 64, variant="int8_per_tensor", device=DEV)
    with pytest.raises(RuntimeError):
        c.prefill(0, e, e)


@pytest.mark.parametrize("variant", ["fp16", "int8_per_token", "int8_per_tensor"])
def test_prefill_under_capture(variant):
    """A captured prefill replayed over new rows in the same buffers, with eager prefills and
    synchronizations in between: each replay equals the eager result."""
    import pa_int8

    tokens, hkv, d = 333, 2, 128
    k, v = (torch.empty(tokens, hkv, d, dtype=torch.float16, device=DEV) for _ in range(2))
    cap, ref = (pa_int8.PagedKVCache(1, hkv, d, 512, variant=variant, device=DEV) for _ in range(2))
    k.normal_(), v.normal_()
    cap.prefill(0, k, v)                      # (warm-up outside the capture)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        cap.prefill(0, k, v)
    for i in range(4):
        g = torch.Generator(device=DEV).manual_seed(i)
        k.normal_(generator=g), v.normal_(generator=g)
        k.mul_(1.0 + i)
        for t in cap._tensors() + ref._tensors():
            t.fill_(5)
        graph.replay()
        torch.cuda.synchronize()
        ref.prefill(0, k, v)
        for a, b in zip(cap._tensors(), ref._tensors()):
            assert torch.equal(bits(a), bits(b)), i
        if variant == "int8_per_tensor":
            assert torch.equal(cap._k_tensor_scale[0], ref._k_tensor_scale[0])
            assert torch.equal(cap._v_tensor_scale[0], ref._v_tensor_scale[0])
