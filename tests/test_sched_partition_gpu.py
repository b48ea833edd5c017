"""GPU tests of the partition that the in-kernel schedule takes from the lengths.

Ragged batches of at most 64 sequences: about four items per resident work-group
whatever the batch (a longer item keeps more softmax weights relative to one running
maximum, and its outputs lie farther from the exact ones).  Equal lengths: the fewest
rounds of one item per CU.  A call that forces the expected partition cuts the same items,
so its output must be the same to the bit; both are also checked against attention
in 64 bits.
"""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
CUS, ITEMS, ITER = 256, 4, 64
SCHED = 2


@pytest.fixture(scope="module", autouse=True)
def _lib(built):
    import pa_int8

    pa_int8.ext()
    yield
    pa_int8.capi().pa_decode_set_schedule(0)


def up(n, step=ITER):
    return -(-n // step) * step


def bounds(int8, head_dim, waves):
    """(shortest ragged item, shortest equal item, longest item) of the schedule."""
    pmin = 1536 if (not int8 and waves == 8) else 2048
    return (pmin if head_dim <= 128 else pmin // 2, 256 * waves // 4,
            (8192 if head_dim <= 128 else 4096) * waves // 4)


def ragged_partition(lens, kv_heads, chunks, int8, head_dim, waves):
    pmin, floor, pmax = bounds(int8, head_dim, waves)
    t = sum(n >> 10 for n in lens)
    part = up(min(math.ceil(t * 1024 * kv_heads / (CUS * 8 // waves * ITEMS)), pmax))
    f = up(min(math.ceil((t + len(lens)) * 1024 * kv_heads * chunks / CUS), pmin))
    return min(min(max(part, max(f, floor)), pmax), up(max(lens)))


def equal_partition(n, seqs, kv_heads, chunks, int8, head_dim, waves):
    _, floor, pmax = bounds(int8, head_dim, waves)
    units = seqs * kv_heads * chunks
    for r in range(1, 5):
        p = up(-(-n // (CUS * r // units)))
        if p <= pmax:
            return min(max(p, floor), up(n))
    raise AssertionError("no partition in four rounds")


def case(lens, heads, kv_heads, d, bs, int8, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    nblk = [-(-n // bs) for n in lens]
    nb = sum(nblk)
    perm = torch.randperm(nb, device=DEV, generator=g).to(torch.int32)
    bt = torch.zeros((len(lens), max(nblk)), dtype=torch.int32, device=DEV)
    at = 0
    for s, k in enumerate(nblk):
        bt[s, :k] = perm[at:at + k]
        at += k
    q = torch.randn(len(lens), heads, d, device=DEV, generator=g).half()
    shapes = (nb, kv_heads, d // 8, bs, 8), (nb, kv_heads, d, bs)
    if int8:
        kc, vc = (torch.randint(-127, 128, s, device=DEV, generator=g, dtype=torch.int8)
                  for s in shapes)
        sc = [0.01 + 0.01 * torch.rand(nb, kv_heads, bs, device=DEV, generator=g) for _ in range(2)]
    else:
        kc, vc = (torch.randn(s, device=DEV, generator=g, dtype=torch.float16) for s in shapes)
        sc = [None, None]
    ctx = torch.tensor(lens, dtype=torch.int32, device=DEV)
    return q, kc, vc, sc, bt, ctx


def run(x, bs, int8, partition=0):
    import pa_int8

    q, kc, vc, sc, bt, ctx = x
    return pa_int8.decode("splitk_int8" if int8 else "splitk", torch.empty_like(q), q, kc, vc, bt,
                          ctx, q.shape[2] ** -0.5, bs, k_scales=sc[0], v_scales=sc[1], check=False,
                          partition_tokens=partition)


def attention64(x, lens, bs):
    q, kc, vc, sc, bt, _ = x
    s, h, d = q.shape
    hkv = kc.shape[1]
    out = torch.empty(s, h, d, dtype=torch.float64, device=DEV)
    for i, n in enumerate(lens):
        blk = bt[i, :-(-n // bs)].long()
        for j in range(hkv):
            k = kc[blk, j].permute(0, 2, 1, 3).reshape(-1, d)[:n].double()
            v = vc[blk, j].permute(0, 2, 1).reshape(-1, d)[:n].double()
            if sc[0] is not None:
                k = k * sc[0][blk, j].reshape(-1)[:n, None].double()
                v = v * sc[1][blk, j].reshape(-1)[:n, None].double()
            hs = slice(j * (h // hkv), (j + 1) * (h // hkv))
            p = torch.softmax(q[i, hs].double() @ k.t().contiguous() * d ** -0.5, -1)
            out[i, hs] = p @ v
    return out


def check(x, lens, bs, int8, want_partition):
    got = run(x, bs, int8)
    same = torch.equal(got, run(x, bs, int8, want_partition))
    assert same, f"not the items of partition {want_partition}"
    ref = attention64(x, lens, bs)
    # the fp16 rounding of the output and of the softmax weights: a quarter to a half of 2^-10
    # each, relative to the result's norm
    err = float((got.double() - ref).norm() / ref.norm())
    assert err <= 2.0 ** -10, err


# (sequences, shortest, longest, heads, kv heads, head_dim, block, int8): rows of one and of
# several head chunks, both group sizes, every width class, shares on both sides of the
# shortest item; the first's items would fill one round when cut at 1.2-1.5 shares
RAGGED = [(24, 900, 9000, 8, 4, 256, 32, False), (24, 900, 9000, 8, 4, 256, 32, True),
          (16, 1000, 8000, 32, 8, 128, 16, False), (16, 1000, 8000, 32, 8, 128, 16, True),
          (20, 2300, 9700, 16, 4, 64, 16, False), (12, 3000, 20000, 32, 1, 256, 16, False),
          (64, 500, 5000, 8, 2, 128, 16, True), (3, 9000, 30000, 64, 4, 128, 16, False),
          (80, 300, 4000, 8, 2, 128, 16, False)]


@pytest.mark.parametrize("seqs,lo,hi,heads,kv_heads,d,bs,int8", RAGGED)
def test_ragged_partition(seqs, lo, hi, heads, kv_heads, d, bs, int8):
    import pa_int8

    g = torch.Generator().manual_seed(seqs + d)
    lens = torch.randint(lo, hi + 1, (seqs,), generator=g).tolist()
    info = plan(seqs, heads, kv_heads, d, bs, -(-max(lens) // bs), int8)
    chunks = heads // kv_heads // info[3]
    pa_int8.capi().pa_decode_set_schedule(SCHED)
    x = case(lens, heads, kv_heads, d, bs, int8)
    check(x, lens, bs, int8, ragged_partition(lens, kv_heads, chunks, int8, d, info[2]))


# equal lengths: units that divide the CUs, that leave a remainder, several head chunks,
# a length that is not a multiple of anything, two and more rounds, the shortest item
EQUAL = [(17, 5001, 12, 2, 128, 16, False), (17, 5001, 12, 2, 128, 16, True),
         (16, 4096, 8, 2, 128, 16, False), (3, 7777, 32, 1, 256, 32, False),
         (5, 40000, 8, 8, 128, 16, True), (64, 9001, 16, 4, 128, 16, True), (2, 700, 8, 1, 8, 16, False)]


@pytest.mark.parametrize("seqs,n,heads,kv_heads,d,bs,int8", EQUAL)
def test_equal_partition(seqs, n, heads, kv_heads, d, bs, int8):
    import pa_int8

    info = plan(seqs, heads, kv_heads, d, bs, -(-n // bs), int8)
    chunks = heads // kv_heads // info[3]
    pa_int8.capi().pa_decode_set_schedule(SCHED)
    x = case([n] * seqs, heads, kv_heads, d, bs, int8)
    check(x, [n] * seqs, bs, int8,
          equal_partition(n, seqs, kv_heads, chunks, int8, d, info[2]))


def plan(seqs, heads, kv_heads, d, bs, blocks, int8):
    """pa_decode_plan_detail of the scheduled launch: (.., .., waves, head tile, ..)."""
    import ctypes

    import pa_int8

    lib = pa_int8.capi()
    assert lib.pa_decode_set_schedule(SCHED) == 0
    info = (ctypes.c_int32 * 7)()
    assert lib.pa_decode_plan_detail(3 if int8 else 1, seqs, heads, d, kv_heads, bs, blocks, 0, 0,
                                     info, 7) == 0
    return list(info)


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("equal", [False, True])
def test_partition_under_a_lowered_row_capacity(equal, int8):
    """The no-alloc entry, whose static scratch holds fewer rows than the schedule asks for
    (eight head chunks of 128 query heads on one kv head): the same items, to the bit."""
    import pa_int8

    lib = pa_int8.capi()
    seqs, heads, d, bs = 17, 128, 256, 16
    g = torch.Generator().manual_seed(5)
    lens = [5001] * seqs if equal else torch.randint(900, 9000, (seqs,), generator=g).tolist()
    kind = 3 if int8 else 1
    info = plan(seqs, heads, 1, d, bs, -(-max(lens) // bs), int8)
    assert heads // info[3] == 8
    assert lib.pa_decode_workspace_bytes(kind, seqs, heads, d, 1, bs, -(-max(lens) // bs), 0,
                                         0) > 64 << 20
    x = case(lens, heads, 1, d, bs, int8)
    q, kc, vc, sc, bt, ctx = x
    if equal:
        want = equal_partition(lens[0], seqs, 1, 8, int8, d, info[2])
    else:
        want = ragged_partition(lens, 1, 8, int8, d, info[2])
    check(x, lens, bs, int8, want)
    out = torch.full_like(q, float("nan"))
    st = lib.pa_paged_decode_attn_noalloc(
        kind, out.data_ptr(), q.data_ptr(), kc.data_ptr(), vc.data_ptr(),
        sc[0].data_ptr() if int8 else None, sc[1].data_ptr() if int8 else None, bt.data_ptr(),
        ctx.data_ptr(), d ** -0.5, bs, seqs, heads, d, 1, kc.shape[0], 8, bt.shape[1], 0, 0,
        torch.cuda.current_stream().cuda_stream)
    assert st == 0, lib.pa_status_string(st)
    same = torch.equal(out, run(x, bs, int8))
    assert same
