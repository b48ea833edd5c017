"""GPU tests of the ops' context-length check (the reference's `min >= 1` rule,
paged_attention_v3_warp.cu:147-148), whose result a kernel writes where the
host polls: positions of the extremes, batches around the reduction's sizes,
work queued before it, calls from several threads and streams in turn (the ops hold the
interpreter's lock, so one call's check ends before the next begins), and the plan that
the lengths choose."""

import threading

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def _lib(built):
    import pa_int8

    pa_int8.ext()


def inputs(n, cap=64, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    blocks = cap // 16
    kc = torch.randn(n * blocks, 1, 1, 16, 8, device=DEV, generator=g).half()
    vc = torch.randn(n * blocks, 1, 8, 16, device=DEV, generator=g).half()
    bt = torch.arange(n * blocks, dtype=torch.int32, device=DEV).view(n, blocks)
    q = torch.randn(n, 1, 8, device=DEV, generator=g).half()
    ctx = torch.randint(1, cap + 1, (n,), device=DEV, generator=g).to(torch.int32)
    return q, kc, vc, bt, ctx


def call(x, variant="warp"):
    import pa_int8

    q, kc, vc, bt, ctx = x
    out = torch.full_like(q, 7)
    pa_int8.VARIANTS[variant](out, q, kc, vc, bt, ctx, 0.3, 16)
    return out


def unchecked(x, variant="warp"):
    import pa_int8

    q, kc, vc, bt, ctx = x
    return pa_int8.decode(variant, torch.empty_like(q), q, kc, vc, bt, ctx, 0.3, 16, check=False)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 256, 257, 1000])
def test_extremes_are_found(n):
    x = inputs(n)
    torch.testing.assert_close(call(x), unchecked(x), rtol=0, atol=0)
    for bad in (0, -5):
        for at in {0, n // 2, n - 1}:
            y = x[:4] + (x[4].clone(),)
            y[4][at] = bad
            out = torch.full_like(x[0], 7)
            import pa_int8
            with pytest.raises(RuntimeError, match="context_lens must be >= 1"):
                pa_int8.VARIANTS["warp"](out, *y, 0.3, 16)
            assert (out == 7).all()      # a refused call leaves its output alone
    torch.testing.assert_close(call(x, "splitk"), unchecked(x, "splitk"), rtol=0, atol=1e-3)


def test_behind_queued_work():
    """The lengths are produced by work that is still queued (longer than the
    check polls before it waits on the stream)."""
    x = inputs(8)
    a = torch.randn(4096, 4096, device=DEV)
    for _ in range(60):
        a = (a @ a) * 1e-3
    late = (x[4].float() + 0 * a[0, 0].nan_to_num()).to(torch.int32)
    torch.testing.assert_close(call(x[:4] + (late,)), unchecked(x), rtol=0, atol=0)


def test_threads_and_streams():
    cases = [inputs(3 + i, seed=i) for i in range(6)]
    want = [unchecked(c) for c in cases]
    torch.cuda.synchronize()
    errors = []

    def work(i):
        try:
            s = torch.cuda.Stream()
            with torch.cuda.stream(s):
                for _ in range(50):
                    got = call(cases[i])
                    s.synchronize()
                    assert torch.equal(got, want[i])
        except Exception as e:       # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[0]


def test_without_host_memory_to_poll():
    """A check that finds no memory to poll reads the lengths back by copy, with the same
    refusals, and the next check polls again."""
    import pa_int8

    x = inputs(8)
    want = unchecked(x)
    slot = pa_int8.ext()._length_slot
    n = slot(0)
    for polled in (1, 0, 1):
        slot(1 - polled)
        assert torch.equal(call(x), want)
        assert slot(0) == n + polled
        n += polled
    bad = x[:4] + (x[4].clone(),)
    bad[4][7] = 0
    out = torch.full_like(x[0], 7)
    slot(1)
    with pytest.raises(RuntimeError, match="context_lens must be >= 1"):
        pa_int8.VARIANTS["warp"](out, *bad, 0.3, 16)
    assert (out == 7).all() and slot(0) == n


def test_read_back_by_copy_chooses_the_same_plan():
    """A check that finds no memory to poll takes the plan that the polled one takes (launches
    above 64 MiB, whose splits show in the last bits)."""
    import pa_int8

    S, H, HKV, D, bs, top = 20, 8, 4, 128, 16, 4100
    lens = [top] + [40 + 97 * i for i in range(S - 1)]
    g = torch.Generator(device=DEV).manual_seed(3)
    nblk = -(-top // bs)
    kc = torch.randn(S * nblk, HKV, D // 8, bs, 8, device=DEV, generator=g).half()
    vc = torch.randn(S * nblk, HKV, D, bs, device=DEV, generator=g).half()
    bt = torch.arange(S * nblk, dtype=torch.int32, device=DEV).view(S, nblk)
    q = torch.randn(S, H, D, device=DEV, generator=g).half()
    slot = pa_int8.ext()._length_slot

    def both(ctx, variant):
        n = slot(0)
        polled = call((q, kc, vc, bt, ctx), variant)
        assert slot(1) == n + 1
        copied = call((q, kc, vc, bt, ctx), variant)
        assert slot(0) == n + 1                      # that one did not poll
        again = call((q, kc, vc, bt, ctx), variant)
        assert slot(0) == n + 2
        assert torch.equal(polled, copied) and torch.equal(polled, again)
        return polled

    ragged = torch.tensor(lens, dtype=torch.int32, device=DEV)
    near = torch.tensor([top - 13 * i for i in range(S)], dtype=torch.int32, device=DEV)
    # (the plans' own outputs differ, so the comparisons above can tell them apart)
    assert not torch.equal(both(ragged, "warp"), unchecked((q, kc, vc, bt, ragged), "warp"))
    assert not torch.equal(both(near, "splitk"), unchecked((q, kc, vc, bt, near), "splitk"))
    both(torch.full_like(near, top), "splitk")
    slot(0)


def test_non_contiguous_lengths_are_still_refused():
    x = inputs(4)
    wide = torch.stack([x[4], x[4]], dim=1)
    with pytest.raises(RuntimeError, match="contiguous"):
        call(x[:4] + (wide[:, 0],))


# lengths whose mean lies below 0.5, above 0.7 and between, of a launch above the 64 MiB
# (bound: every sequence at the longest) from which the lengths choose the plan; the choice
# itself is pinned on the CPU (test_host.py), here each kind's call must be the launch it names
@pytest.mark.parametrize("pattern", ["ragged", "near_equal", "between", "equal"])
@pytest.mark.parametrize("variant", ["warp", "splitk", "warp_int8", "splitk_int8"])
def test_every_plan_gives_the_same_attention(pattern, variant):
    import pa_int8

    S, H, HKV, D, bs, top = 20, 8, 4, 128, 16, 4100
    lens = {"ragged": [top] + [40 + 97 * i for i in range(S - 1)],
            "near_equal": [top - 13 * i for i in range(S)],
            "between": [1000 if i % 2 else top for i in range(S)],
            "equal": [top] * S}[pattern]
    mean = sum(lens) // S
    assert {"ragged": 2 * mean < top, "near_equal": 0.7 * top <= mean < top,
            "between": top <= 2 * mean and mean < 0.7 * top, "equal": mean == top}[pattern]
    g = torch.Generator(device=DEV).manual_seed(len(pattern))
    nblk = -(-top // bs)
    nb = S * nblk
    bt = torch.randperm(nb, device=DEV, generator=g).to(torch.int32).view(S, nblk)
    q = torch.randn(S, H, D, device=DEV, generator=g).half()
    ctx = torch.tensor(lens, dtype=torch.int32, device=DEV)
    int8 = variant.endswith("int8")
    if int8:
        kc = torch.randint(-127, 128, (nb, HKV, D // 8, bs, 8), device=DEV, generator=g).to(torch.int8)
        vc = torch.randint(-127, 128, (nb, HKV, D, bs), device=DEV, generator=g).to(torch.int8)
        ks, vs = (0.01 + 0.02 * torch.rand(nb, HKV, bs, device=DEV, generator=g) for _ in range(2))
        extra = (ks, vs)
    else:
        kc = torch.randn(nb, HKV, D // 8, bs, 8, device=DEV, generator=g).half()
        vc = torch.randn(nb, HKV, D, bs, device=DEV, generator=g).half()
        ks = vs = None
        extra = ()
    ops = pa_int8.VARIANTS_INT8 if int8 else pa_int8.VARIANTS
    got = ops[variant](torch.empty_like(q), q, kc, vc, *extra, bt, ctx, 0.09, bs)
    other = variant.replace("warp", "splitk") if "warp" in variant else variant.replace("splitk", "warp")
    launched = {"ragged": "splitk", "near_equal": "warp", "equal": "warp"}.get(pattern)
    launched = variant if launched is None else launched + ("_int8" if int8 else "")
    for name in (variant, other):
        want = pa_int8.decode(name, torch.empty_like(q), q, kc, vc, bt, ctx, 0.09, bs, k_scales=ks,
                              v_scales=vs, check=False)
        # (the two plans cut the lengths differently, which shows in the last bits)
        assert torch.equal(got, want) == (name == launched), (name, launched)
        # both round an fp32 result to fp16: two roundings apart, and the fp16 softmax
        # weights of differently cut splits (2^-11 each, averaged over the tokens)
        torch.testing.assert_close(got.float(), want.float(), rtol=4e-3, atol=1e-3)
