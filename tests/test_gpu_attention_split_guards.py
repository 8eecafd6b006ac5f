"""fp32 attention on the fp16 matrix pipe: results that a scale taken from other values has left too few bits, each row and each column for itself.

Bounds: 4e-6 of a row's 2-norm (fp32 logits, probabilities and sums of up to 1100 terms; such rows show up to 1e-6), times an eighth of the largest
visible logit where that is above eight, since 2^-24 of a logit is a relative error of its probability."""
import math

import pytest
import torch

from _util import kernels_of

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    from aidotnet.tensors_amd import Mi355Engine
    return Mi355Engine()


def randn(seed, *shapes):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(*s, device="cuda", generator=gen) for s in shapes]


def reference(q, k, v, hidden=None):
    s = torch.matmul(q.double(), k.double().transpose(2, 3).contiguous()) / math.sqrt(q.shape[-1])
    if hidden is not None:
        s = s.masked_fill(hidden, -math.inf)
    p = torch.softmax(s, -1)
    return torch.matmul(p, v.double()), p, s.masked_fill(s == -math.inf, 0.0).abs().amax()


def worst_row(got, want):
    return float(((got.double() - want).norm(dim=-1) / want.norm(dim=-1)).nan_to_num(math.inf).max())


def later(Sq, Sk, offset=0):
    return torch.arange(Sk, device="cuda")[None, :] > torch.arange(Sq, device="cuda")[:, None] + offset


# one range of the keys, several of them; workgroups of one, two and four key groups
SHAPES = [(70, 70, 32), (200, 200, 64), (40, 200, 64), (130, 300, 128), (40, 1000, 32), (40, 1000, 64), (40, 1000, 128)]


@pytest.mark.parametrize("size", [1e6, 1e10, 1e30])
@pytest.mark.parametrize("option", ["padding", "plane", "causal", "range"])
@pytest.mark.parametrize("Sq,Sk,D", SHAPES)
def test_large_values_out_of_sight(eng, Sq, Sk, D, option, size):
    """V far larger at keys that a row does not see, in its first tile among others."""
    q, k, v = randn(Sk + D, (1, 2, Sq, D), (1, 2, Sk, D), (1, 2, Sk, D))
    if option in ("padding", "plane"):
        hidden = torch.zeros(1, 1, 1 if option == "padding" else Sq, Sk, dtype=torch.bool, device="cuda")
        hidden[..., 20:29] = True
        hidden[..., Sk - 9:] = True
        v[:, :, 20:29] *= size
        v[:, :, Sk - 9:] *= size
        want, _, _ = reference(q, k, v, hidden)
        o, _ = eng.ScaledDotProductAttention(q, k, v, ~hidden, returnWeights=False)
        assert worst_row(o, want) <= 4e-6
        return
    offset = Sk - Sq if option == "range" else 0
    v[:, :, offset + min(Sq, Sk) // 2:] *= size              # from the middle query's diagonal on
    want, _, _ = reference(q, k, v, later(Sq, Sk, offset))
    o, _ = eng.FlashAttention(q, k, v, isCausal=True, queryOffset=offset)
    assert worst_row(o, want) <= 4e-6


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("Sq,Sk", [(200, 200), (40, 1000)])
@pytest.mark.parametrize("small", [1.0, 1e-3])
def test_sharp_probabilities_over_a_first_tile_of_zeros(eng, small, Sq, Sk, D):
    """A left-padded cache: the first tiles of V give no scale; each row's weight lies on a few of the keys behind them."""
    q, k, v = randn(Sk + D, (1, 4, Sq, D), (1, 4, Sk, D), (1, 4, Sk, D))
    q *= 8
    v *= small
    v[:, :, :130] = 0.0
    hidden = torch.zeros(1, 1, 1, Sk, dtype=torch.bool, device="cuda")
    hidden[..., :130] = True
    want, _, big = reference(q, k, v)
    o, _ = eng.FlashAttention(q, k, v)
    seen = want.norm(dim=-1) > 1e-3 * small                   # (rows whose weight lies on the zeros have nothing left but their tails)
    assert float(((o.double() - want).norm(dim=-1) / want.norm(dim=-1))[seen].max()) <= 4e-6 * max(1.0, float(big) / 8)
    want, _, big = reference(q, k, v, hidden)
    o, _ = eng.ScaledDotProductAttention(q, k, v, ~hidden, returnWeights=False)
    assert worst_row(o, want) <= 4e-6 * max(1.0, float(big) / 8)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("Sk", [200, 1000])
def test_weight_far_below_the_largest(eng, Sk, D):
    """One key takes nearly all of the weight and carries almost nothing: the rows are sums of probabilities of 2^-14."""
    q, k, v = randn(Sk + D, (1, 2, 40, D), (1, 2, Sk, D), (1, 2, Sk, D))
    q[..., 0] = 8.0
    k[..., 0] = 0.0
    k[:, :, 3, 1:] = 0.0
    k[:, :, 3, 0] = 14 * math.log(2) * math.sqrt(D) / 8
    v[:, :, 3] *= 2e-3
    want, _, big = reference(q, k, v)
    o, _ = eng.FlashAttention(q, k, v)
    assert worst_row(o, want) <= 4e-6 * max(1.0, float(big) / 8)


@pytest.mark.parametrize("D", [32, 64, 128])
def test_one_far_lower_logit(eng, D):
    """Visible keys whose logits are far below all others set the scales of Q and K, and do not vouch for the others' logits."""
    q, k, v = randn(D, (1, 2, 40, D), (1, 2, 200, D), (1, 2, 200, D))
    q[..., 0] = 1e7
    k[..., 0] = 0.0
    k[:, :, 7::16, 0] = -1e7
    s = torch.matmul(q.double(), k.double().transpose(2, 3).contiguous()) / math.sqrt(D)
    want = torch.matmul(torch.softmax(s, -1), v.double())
    o, _ = eng.FlashAttention(q, k, v)
    assert worst_row(o, want) <= 4e-6


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("Sk", [300, 1600])
@pytest.mark.parametrize("size", [1e38, 3.3e38])
def test_values_at_the_upper_end_of_a_later_tile(eng, size, Sk, D):
    q, k, v = randn(Sk + D, (1, 2, 40, D), (1, 2, Sk, D), (1, 2, Sk, D))
    q[..., 0] = 30.0
    k[..., 0] = 0.0
    k[:, :, 250, 0] = 30.0
    v[:, :, 250] = size * torch.sign(v[:, :, 250])
    want, _, big = reference(q, k, v)
    o, _ = eng.FlashAttention(q, k, v)
    assert bool(o.isfinite().all()) and worst_row(o, want) <= 4e-6 * max(1.0, float(big) / 8)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("Sk", [300, 1600])
@pytest.mark.parametrize("size", [1e-33, 1e-35])
def test_values_at_the_lower_end(eng, size, Sk, D):
    """(numbers below 1.2e-38 have fewer bits: half a unit of 2^-149 of each result is granted)"""
    q, k, v = randn(Sk + D, (1, 2, 40, D), (1, 2, Sk, D), (1, 2, Sk, D))
    v *= size
    want, _, _ = reference(q, k, v)
    o, _ = eng.FlashAttention(q, k, v)
    assert worst_row(o, want) <= 4e-6 + math.sqrt(D) * 2.0 ** -149 / float(want.norm(dim=-1).min())


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("case", ["zero rows", "small", "zero rows, padded"])
def test_probabilities_of_vanishing_logits(eng, case, D):
    """Rows of zeros, and products below the range of fp32: equal probabilities, zeros above the diagonal."""
    q, k, v = randn(D, (1, 2, 100, D), (1, 2, 100, D), (1, 2, 100, D))
    if case == "small":
        q, k = q * 1e-20, k * 1e-20
    else:
        q[:, :, ::3] = 0.0
        k *= 1e-5
    hidden, mask = later(100, 100), None
    if case == "zero rows, padded":
        hidden = torch.zeros(1, 1, 1, 100, dtype=torch.bool, device="cuda")
        hidden[..., 40:50] = True
        mask = ~hidden
    want, p, _ = reference(q, k, v, hidden)
    o, w = eng.ScaledDotProductAttention(q, k, v, mask, isCausal=mask is None)
    assert worst_row(o, want) <= 4e-6 and worst_row(w, p) <= 4e-6
    assert bool((w[hidden.expand_as(w)] == 0).all())


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("hidden_key", [False, True])
def test_columns(eng, hidden_key, D):
    """A column of zeros and one far below the others, or far below them but at keys that no row sees."""
    q, k, v = randn(D, (1, 2, 200, D), (1, 2, 200, D), (1, 2, 200, D))
    v[..., 1] = 0.0
    v[..., 5] *= 1e-9
    hidden, mask = None, None
    if hidden_key:
        hidden = torch.zeros(1, 1, 1, 200, dtype=torch.bool, device="cuda")
        hidden[..., 30:34] = True
        mask = ~hidden
        v[:, :, 30:34, 5] = 1.0
    want, _, _ = reference(q, k, v, hidden)
    o, _ = eng.ScaledDotProductAttention(q, k, v, mask, returnWeights=False)
    assert float((o[..., 5].double() - want[..., 5]).norm() / want[..., 5].norm()) <= 4e-6
    assert bool((o[..., 1] == 0).all())


@pytest.mark.parametrize("D", [32, 64, 128])
def test_general_kernel_on_request(D):
    """The switch that routes every attention shape through the general kernel reaches fp32, its key ranges and its probabilities."""
    from aidotnet.tensors_amd import Mi355Backend, Mi355Engine
    be = Mi355Backend()
    eng = Mi355Engine(be)
    q, k, v = randn(D, (1, 2, 40, D), (1, 2, 1000, D), (1, 2, 1000, D))
    call = lambda: eng.ScaledDotProductAttention(q, k, v)
    o, w = call()
    assert [n.split("<")[0] for n in kernels_of(call)] == ["attn_split_kernel", "attn_split_merge_kernel", "attn_weights_split_kernel"]
    be.SetAttentionFastPath(False)
    names = kernels_of(call)
    assert [n.split("<")[0] for n in names] == ["attn_fwd_kernel", "attn_weights_kernel"], names
    o2, w2 = call()
    assert float((o - o2).norm() / o2.norm()) <= 4e-6 and float((w - w2).norm() / w2.norm()) <= 4e-6


def versus_general_kernel(call, exact):
    """Error of each output of `call` against float64 in the 2-norm, as chosen and on the general kernel (fp32 pipe)."""
    from aidotnet.tensors_amd import Mi355Backend, Mi355Engine
    be = Mi355Backend()
    eng = Mi355Engine(be)
    found = []
    for fast in (True, False):
        be.SetAttentionFastPath(fast)
        found.append([float((got.double() - want).norm() / want.norm()) for got, want in zip(call(eng), exact)])
    return list(zip(*found))


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("B,H,Sq,Sk,D", [(8, 12, 512, 512, 64), (2, 16, 200, 200, 32), (4, 16, 300, 300, 128), (1, 8, 1024, 1024, 128), (1, 8, 200, 1000, 64)])
def test_log_sum_is_as_exact_as_on_the_fp32_pipe(B, H, Sq, Sk, D, causal):
    """(4.1e-8 where the fp32 pipe has 5.0e-8; the margin is for what two sums of some ten thousand errors differ by)"""
    q, k, v = randn(Sk + D, (B, H, Sq, D), (B, H, Sk, D), (B, H, Sk, D))
    s = torch.matmul(q.double(), k.double().transpose(2, 3).contiguous()) / math.sqrt(D)
    lse = torch.logsumexp(s.masked_fill(later(Sq, Sk), -math.inf) if causal else s, -1)
    (chosen, general), = versus_general_kernel(lambda eng: [eng.FlashAttention(q, k, v, isCausal=causal)[1]], [lse])
    assert chosen <= 1.03 * general


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("B,H,Sq,Sk,D", [(2, 16, 100, 100, 32), (3, 16, 139, 149, 32), (4, 12, 512, 512, 64), (5, 12, 166, 166, 128), (1, 8, 64, 1000, 64)])
def test_probabilities_are_as_exact_as_on_the_fp32_pipe(B, H, Sq, Sk, D, causal):
    """(0.74 to 0.94 of the fp32 pipe's error, which is that of exponents of five to ten)"""
    q, k, v = randn(Sk + D, (B, H, Sq, D), (B, H, Sk, D), (B, H, Sk, D))
    want, p, _ = reference(q, k, v, later(Sq, Sk, Sk - Sq) if causal else None)
    results = versus_general_kernel(lambda eng: eng.ScaledDotProductAttention(q, k, v, isCausal=causal), [want, p])
    for chosen, general in results:
        assert chosen <= 1.02 * general, results


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("D,Sk", [(8, 16), (8, 64), (8, 128), (8, 129), (8, 256), (8, 432), (8, 433), (16, 16), (16, 32), (16, 64), (16, 65), (16, 176), (16, 177), (24, 90), (24, 91),
                                  (32, 16), (32, 32), (32, 33), (32, 48), (32, 49), (80, 16), (128, 16)])
def test_few_keys_are_as_exact_as_on_the_fp32_pipe(D, Sk, causal):
    """Both sides of the lines up to which few keys and narrow heads stay on the fp32 pipe (two sums of errors over 30000 results differ by 2 %)."""
    q, k, v = randn(Sk + D, (4, 32, Sk, D), (4, 32, Sk, D), (4, 32, Sk, D))
    want, _, _ = reference(q, k, v, later(Sk, Sk) if causal else None)
    (chosen, general), = versus_general_kernel(lambda eng: [eng.FlashAttention(q, k, v, isCausal=causal)[0]], [want])
    assert chosen <= 1.03 * general


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("option", ["padding", "plane"])
def test_large_logits_under_a_mask(eng, option, D):
    """Logits of thousands: rows whose largest one is far from zero are held, those that see one key of little weight are not."""
    q, k, v = randn(D, (1, 2, 100, D), (1, 2, 200, D), (1, 2, 200, D))
    q, k = q * 60, k * 60
    q[:, :, 7] *= 1e-4
    hidden = torch.zeros(1, 1, 1 if option == "padding" else 100, 200, dtype=torch.bool, device="cuda")
    hidden[..., :50] = True
    want, _, big = reference(q, k, v, hidden)
    o, _ = eng.ScaledDotProductAttention(q, k, v, ~hidden, returnWeights=False)
    # (2^-24 of a logit is a relative error of its probability)
    assert float((o.double() - want).norm() / want.norm()) <= 1.5e-6 * max(1.0, float(big) / 4)
    assert worst_row(o[:, :, 7], want[:, :, 7]) <= 4e-6


@pytest.mark.parametrize("D", [32, 64, 128])
def test_column_beyond_the_last_row(eng, D):
    """Keys behind the last row's diagonal, which the idle rows of its wave would see, do not vouch for a column."""
    q, k, v = randn(D, (1, 2, 20, D), (1, 2, 400, D), (1, 2, 400, D))
    v[:, :, :120, 5] *= 1e-9
    want, _, _ = reference(q, k, v, later(20, 400, 100))
    o, _ = eng.FlashAttention(q, k, v, isCausal=True, queryOffset=100)
    assert float((o[..., 5].double() - want[..., 5]).norm() / want[..., 5].norm()) <= 4e-6


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("first,end", [(300, 310), (320, 340), (300, 500)])
def test_large_values_in_one_key_group(eng, first, end, D):
    """Key groups and ranges without the large values hold next to nothing of a row: that alone is no reason to compute it again (whose sums, as those of
    the fp32 pipe, would leave the range of fp32)."""
    q, k, v = randn(7, (1, 2, 40, D), (1, 2, 1600, D), (1, 2, 1600, D))
    v = v.clamp(-2, 2)
    v[:, :, first:end] *= 1.5e38
    want, _, _ = reference(q, k, v)
    o, _ = eng.FlashAttention(q, k, v)
    assert bool(o.isfinite().all()) and worst_row(o, want) <= 4e-6


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("option", ["plain", "plane", "causal"])
def test_probabilities_of_large_logits(eng, option, D):
    """Logits of thousands: both passes form them on the same pipe, or a probability of one is off by the error of either (2 to 9 times the fp32 pipe's).
    (0.7 to 1.16 of it; what is left are the few rows whose two largest logits nearly tie, whose errors two pipes draw differently)"""
    q, k, v = randn(D, (1, 4, 200, D), (1, 4, 200, D), (1, 4, 200, D))
    q, k = q * 60, k * 60
    hidden = later(200, 200) if option == "causal" else (randn(D + 1, (1, 1, 200, 200))[0] < -0.5) if option == "plane" else None
    want, p, _ = reference(q, k, v, hidden)
    (o, _), (chosen, general) = versus_general_kernel(lambda eng: eng.ScaledDotProductAttention(q, k, v, ~hidden if option == "plane" else None, isCausal=option == "causal"), [want, p])
    assert chosen <= 1.3 * general


@pytest.mark.parametrize("Sq,Sk", [(200, 200), (40, 1000)])
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("option", ["plain", "padding"])
@pytest.mark.parametrize("case", ["column", "first tile", "row"])
def test_probabilities_beside_a_second_computation(eng, case, option, D, Sq, Sk):
    """Where V or another row has the results computed again on the fp32 pipe, a row's probabilities and its sum are still of one pipe (apart, 2 to 5 times
    the fp32 pipe's error over logits of deviation 64, 7 over 3600; bound as above)."""
    for size in (8, 60):
        q, k, v = randn(D, (1, 4, Sq, D), (1, 4, Sk, D), (1, 4, Sk, D))
        q, k = q * size, k * size
        if case == "column":
            v[..., 3] *= 1e-12
        elif case == "first tile":                              # far larger values at keys of no weight
            v[:, :, :64] *= 1e12
            k[:, :, :64, 1] = -1000.0 * size
            q[..., 1] = size
        else:                                                   # one row of small logits under a coarse scale
            k[..., 0] = 0
            q[:, :, 5] = 0
            q[:, :, 5, 0] = size
        hidden = None
        if option == "padding":
            hidden = torch.zeros(1, 1, 1, Sk, dtype=torch.bool, device="cuda")
            hidden[..., Sk - 20:] = True
        _, p, _ = reference(q, k, v, hidden)
        (chosen, general), = versus_general_kernel(lambda eng: [eng.ScaledDotProductAttention(q, k, v, None if hidden is None else ~hidden)[1]], [p])
        assert chosen <= 1.3 * general, (size, chosen, general)
