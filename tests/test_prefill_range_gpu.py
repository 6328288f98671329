"""The pipelined prefill kernel: scores that leave the range of an item's first reference (rows whose later
keys score hundreds above the first 64, far below them, or both, with overflow to infinity on the way; the
softmax is then close to one-hot, and the fp32 oracle gives it), the merge of its splits, the range of V,
rows past a sequence's end, and the edges of steps and tiles.

Which kernel a call takes follows from its launch bounds (small_prefill); a key-count bound of BOUND_K
takes any call of this file to the pipelined one."""
import pytest
import torch

import oracle
import pagedkv
from paged_helpers import assert_close_bf16

pytestmark = pytest.mark.gpu
D = 128
BOUND_K = 1 << 21
GROUPS = [(16, 8), (4, 4), (8, 2), (8, 1)]  # GQA groups 2, 1, 4, 8


def _batch(seqs, hq, hkv, steps, seed):
    """q and k whose products follow `steps`: key t of every sequence scores 16 steps(t) D^-0.5 more
    than small noise (exact in bf16 for whole steps up to 256)."""
    g = torch.Generator().manual_seed(seed)
    nq, nk = sum(q for q, _ in seqs), sum(k for _, k in seqs)
    q = 0.25 * torch.randn(nq, hq, D, generator=g)
    k = 0.25 * torch.randn(nk, hkv, D, generator=g)
    q[..., 0] = 16.0
    k[..., 0] = torch.cat([torch.tensor([float(steps(t, n)) for t in range(n)]) for _, n in seqs])[:, None]
    v = torch.randn(nk, hkv, D, generator=g)
    return (x.to(torch.bfloat16) for x in (q, k, v))


def _paged(seqs, k, v, width, bs=64):
    """Caches and a block table of `width` blocks a sequence; every row that holds no key is NaN."""
    hkv, blocks = k.shape[1], sum(-(-n // bs) for _, n in seqs)
    order = torch.randperm(blocks, generator=torch.Generator().manual_seed(1)).tolist()
    kc, vc = (torch.full((blocks, bs, hkv, D), float("nan"), dtype=torch.bfloat16) for _ in range(2))
    bt = torch.full((len(seqs), width), -1, dtype=torch.int32)
    lo = 0
    for b, (_, n) in enumerate(seqs):
        for j in range(-(-n // bs)):
            blk, m = order.pop(), min(bs, n - j * bs)
            bt[b, j] = blk
            kc[blk, :m], vc[blk, :m] = k[lo + j * bs:lo + j * bs + m], v[lo + j * bs:lo + j * bs + m]
        lo += n
    return kc, vc, bt


def _run(gpu, q, k, v, seqs, paged, causal=True, bound=BOUND_K):
    """The call over a paged copy of k and v, or flat with NaN rows behind the last one (inside the
    allocation): a row read past a sequence's end makes its tile's outputs NaN."""
    hq, hkv, max_q = q.shape[1], k.shape[1], max(a for a, _ in seqs)
    max_k = bound or max(b for _, b in seqs)
    if bound:  # an estimate of 36 tiles per work-group of 256, as small_prefill makes it
        keys = max_k if paged else (max_k + sum(a for a, _ in seqs) / len(seqs)) / 2
        keys = (keys + 256 * hkv // hq) / 2 if causal else keys
        assert sum(a for a, _ in seqs) * keys * hkv >= 36 * 256 * (256 * hkv // hq) * 64
    cu_q, cu_k = _cu([a for a, _ in seqs]).to(gpu), _cu([b for _, b in seqs]).to(gpu)
    if paged:
        kd, vd, bt = (x.to(gpu) for x in _paged(seqs, k, v, -(-max_k // 64)))
    else:
        pad, bt = torch.full((128, hkv, D), float("nan"), dtype=torch.bfloat16), None
        kd, vd = (torch.cat([x, pad]).to(gpu)[:len(x)] for x in (k, v))
    out = pagedkv.varlen_attention(q.to(gpu), kd, vd, cu_q, cu_k, max_q, max_k, D ** -0.5, causal, bt)
    torch.cuda.synchronize()
    return out.cpu()


def _cu(lens):
    return torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)


def _oracle(q, k, v, seqs, causal=True):
    return oracle.varlen_attention(q, k, v, _cu([a for a, _ in seqs]), _cu([b for _, b in seqs]), D ** -0.5, causal, None)


def _check(gpu, q, k, v, seqs, what, paged=True, causal=True, bound=BOUND_K, scale_out=1.0):
    """_run against the oracle (scale_out: a power of two that brings the outputs near 1)."""
    out = _run(gpu, q, k, v, seqs, paged, causal, bound)
    assert_close_bf16(out.float() * scale_out, _oracle(q, k, v, seqs, causal).float() * scale_out, what)
    return out


STEPS = {
    "jump": lambda t, n: 150 if t >= 80 else 0,                 # 212 nats above the first keys
    "late": lambda t, n: 100 if t == n - 1 else 0,              # one key, at the end
    "ramp": lambda t, n: min(240, t // 8),                      # up to 339 nats, step by step
    "fall": lambda t, n: -200 if t >= 64 else 0,                # everything after the first tile vanishes
    "low": lambda t, n: -250 if t < 64 else 0,                  # the first tile vanishes
    "inside": lambda t, n: 50 if t % 96 == 70 else 0,           # 71 nats: inside the headroom
}


@pytest.mark.parametrize("steps", list(STEPS))
@pytest.mark.parametrize("hq,hkv", GROUPS)
@pytest.mark.parametrize("paged", [True, False])
@pytest.mark.parametrize("bound", [0, BOUND_K])
def test_scores_beyond_the_first_reference(gpu, bound, steps, hq, hkv, paged):
    # bound 0: the lengths' own bounds, which take some of the groups to the eight-wavefront kernel
    seqs = [(130, 700), (2, 65), (33, 2000), (257, 257), (1100, 1500), (40, 40)] if paged else \
        [(130, 130), (2, 2), (1800, 1800), (65, 65), (3, 3), (300, 300)]
    print(f"[prefill-range] {steps} hq={hq} hkv={hkv} paged={paged} bound={bound}", flush=True)
    _check(gpu, *_batch(seqs, hq, hkv, STEPS[steps], 7), seqs, f"{steps} paged={paged}", paged, bound=bound)


@pytest.mark.parametrize("large", [False, True])
@pytest.mark.parametrize("tail", [1, 31, 32, 33, 63, 64, 65, 127, 128, 129, 191, 192, 193, 320])
def test_step_and_tile_edges(gpu, tail, large):
    """Key counts around the 32-key steps, the tiles and the depth of the tile pipeline."""
    seqs = [(max(2, tail), tail + 1), (2, tail + 1), (64, tail + 64), (127, tail + 130)]
    print(f"[prefill-range] edges tail={tail}", flush=True)
    _check(gpu, *_batch(seqs, 8, 4, lambda t, n: 0, tail), seqs, f"tail {tail}", False, bound=BOUND_K if large else 0)


@pytest.mark.parametrize("paged", [True, False])
@pytest.mark.parametrize("hq,hkv", GROUPS)
@pytest.mark.parametrize("keys", [63, 65, 127, 129, 191, 193, 255, 257, 319, 321, 383, 449])
def test_last_tile_of_short_items(gpu, keys, hq, hkv, paged):
    """Items of 1 to 8 tiles whose last tile ends with the sequence, as the last of a flat batch and,
    paged, behind a cached prefix too."""
    print(f"[prefill-range] last tile keys={keys} hq={hq} hkv={hkv} paged={paged}", flush=True)
    seqs = [(1500, 1500)] + ([(60, keys), (2, keys)] if paged else []) + [(keys, keys)]
    _check(gpu, *_batch(seqs, hq, hkv, lambda t, n: 0, 11), seqs, f"keys={keys} paged={paged}", paged)


@pytest.mark.parametrize("paged", [True, False])
@pytest.mark.parametrize("hq,hkv", GROUPS)
def test_rows_and_items_without_keys(gpu, hq, hkv, paged):
    """Fewer keys than query rows: rows before the first key are 0, whole items have no tile."""
    print(f"[prefill-range] without keys hq={hq} hkv={hkv} paged={paged}", flush=True)
    seqs = [(300, 200), (40, 3000), (700, 20), (90, 90)]
    out = _check(gpu, *_batch(seqs, hq, hkv, lambda t, n: 0, 12), seqs, "rows without keys", paged)
    assert torch.count_nonzero(out[:100].float()) == 0
    assert torch.count_nonzero(out[340:340 + 680].float()) == 0


@pytest.mark.parametrize("paged", [True, False])
@pytest.mark.parametrize("hq,hkv", GROUPS)
@pytest.mark.parametrize("steps", ["none", "jump", "fall"])
def test_not_causal(gpu, steps, hq, hkv, paged):
    print(f"[prefill-range] not causal {steps} hq={hq} hkv={hkv} paged={paged}", flush=True)
    seqs = [(130, 700), (2, 65), (33, 1333), (257, 130), (40, 40)]
    fn = STEPS.get(steps, lambda t, n: 0)
    _check(gpu, *_batch(seqs, hq, hkv, fn, 13), seqs, f"not causal {steps}", paged, causal=False)


@pytest.mark.parametrize("order", ["rise first", "rise last"])
@pytest.mark.parametrize("steps", [20, 40, 56, 58, 60, 62])
@pytest.mark.parametrize("hq,hkv", GROUPS)
def test_merge_weighs_splits_by_their_sums(gpu, hq, hkv, steps, order):
    """Two splits of one unit whose weights differ by 8 to 1 while their references lie far apart: in one
    the two heavy keys come late (2 log2 per step above its first keys), in the other among the first
    64, two steps higher."""
    print(f"[prefill-range] merge hq={hq} hkv={hkv} steps={steps} {order}", flush=True)
    late, early = (0, 512) if order == "rise first" else (512, 0)
    heavy = {late + 100: steps, late + 300: steps, early + 8: steps + 2}
    seqs = [(40, 1024)]     # 16 tiles: two splits of 8
    _check(gpu, *_batch(seqs, hq, hkv, lambda t, n: heavy.get(t, 0), 5), seqs, f"{steps} {order}")


@pytest.mark.parametrize("hq,hkv", GROUPS)
@pytest.mark.parametrize("key", [5, 40, 70, 130, 500])
def test_one_heavy_key_gives_its_value_exactly(gpu, hq, hkv, key):
    """A key 40 log2 above all others: numerator and denominator weigh it by the same rounded p, so every row
    is its V row, bit for bit, whatever the fraction that p was rounded from."""
    print(f"[prefill-range] heavy key={key} hq={hq} hkv={hkv}", flush=True)
    seqs = [(100, 560), (300, 560)]
    q, k, v = _batch(seqs, hq, hkv, lambda t, n: 20 if t == key else 0, 3 + key)
    out = _check(gpu, q, k, v, seqs, f"key {key}")
    seen = torch.cat([torch.arange(a) + b - a >= key for a, b in seqs])
    rows = torch.cat([torch.full((a,), i) for i, (a, _) in enumerate(seqs)]) * 560 + key
    assert torch.equal(out[seen], v[rows][seen].repeat_interleave(hq // hkv, 1))


@pytest.mark.parametrize("steps", [0, 30, 55])
@pytest.mark.parametrize("exponent", [-100, -70, 70, 110])
@pytest.mark.parametrize("hq,hkv", GROUPS)
def test_values_of_any_magnitude(gpu, hq, hkv, exponent, steps):
    """V rows far from 1 beside scores that rise by up to 112 log2 over an item: neither the products p v nor
    their sums may leave the range of fp32 where the output does not."""
    print(f"[prefill-range] V 2^{exponent} steps={steps} hq={hq} hkv={hkv}", flush=True)
    seqs = [(130, 700), (300, 333)]
    q, k, v = _batch(seqs, hq, hkv, lambda t, n: steps if t % 90 == 77 else 0, 9)
    v = (v.float() * 2.0 ** exponent).to(torch.bfloat16)
    _check(gpu, q, k, v, seqs, f"V 2^{exponent}, steps {steps}", scale_out=2.0 ** -exponent)


@pytest.mark.parametrize("hq,hkv", GROUPS)
def test_first_keys_of_minus_infinity(gpu, hq, hkv):
    """The first 64 keys score -infinity (bf16's lowest value in K), the others so low that without a reference
    of their own 2^score is below fp32's normal range for most of them."""
    print(f"[prefill-range] -inf first hq={hq} hkv={hkv}", flush=True)
    seqs = [(230, 300)]     # every row sees more than 64 keys
    q, k, v = _batch(seqs, hq, hkv, lambda t, n: -61 if t == 67 else -62, 4)
    k[:64, :, 0] = torch.finfo(torch.bfloat16).min
    _check(gpu, q, k, v, seqs, "-inf first")


@pytest.mark.parametrize("steps", ["none", "jump", "ramp"])
@pytest.mark.parametrize("prefix", [0, 16, 48])
@pytest.mark.parametrize("hq,hkv", GROUPS)
def test_non_finite_values_stay_behind_the_causal_limit(gpu, hq, hkv, prefix, steps):
    """NaN and infinities in a V row reach rows whose block of 32 ends in an earlier 64-key tile in no way, also
    where the scores need a running maximum."""
    print(f"[prefill-range] non-finite V hq={hq} hkv={hkv} prefix={prefix} {steps}", flush=True)
    lq, bad = 700, 330
    seqs = [(lq, lq + prefix)]
    q, k, v = _batch(seqs, hq, hkv, STEPS.get(steps, lambda t, n: 0), 8)
    hot = v.clone()
    hot[bad, :, ::2] = float("nan")
    hot[bad, :, 1::2] = float("inf")
    out = _run(gpu, q, k, hot, seqs, True)
    last = torch.arange(lq) // 32 * 32 + 31 + prefix      # the last key that a row's block of 32 sees
    clean = last < bad // 64 * 64
    assert clean.sum() > 200
    assert_close_bf16(out[clean], _oracle(q, k, v, seqs)[clean], "rows before the non-finite key")
    assert not out[bad + 64 - prefix:].isfinite().any()


@pytest.mark.parametrize("paged", [True, False])
@pytest.mark.parametrize("hq,hkv", GROUPS)
def test_both_kernels_round_alike(gpu, hq, hkv, paged):
    """The pipelined and the eight-wavefront kernel take the same reference and the same rounded p: their
    outputs differ only where the order of a row's sum moves a result across a rounding boundary of bf16
    (fp32 sums of up to 1000 terms: about 2^-20 of a bf16 step of 2^-9, so one output in some thousand)."""
    print(f"[prefill-range] both kernels hq={hq} hkv={hkv} paged={paged}", flush=True)
    seqs = [(130, 700), (40, 1000), (2, 66)] if paged else [(300, 300), (65, 65), (2, 2)]
    g = torch.Generator().manual_seed(17)
    nq, nk = sum(a for a, _ in seqs), sum(b for _, b in seqs)
    q, k, v = (torch.randn(n, h, D, generator=g).to(torch.bfloat16) for n, h in ((nq, hq), (nk, hkv), (nk, hkv)))
    small, large = (_run(gpu, q, k, v, seqs, paged, bound=b) for b in (0, BOUND_K))
    same = (small.view(torch.int16) == large.view(torch.int16)).float().mean().item()
    print(f"equal: {same:.5f}", flush=True)
    assert same >= 0.998
