"""Token sampler kernel (ph_sample_top_p through kernels.sample_top_p) against the float64 oracle
(oracle/ref_sampler.py, after parrot/engine/builtin/models/sampler.py:19-66).

Token ids are integers, so the comparison is exact -- on every row whose decision is not within rounding noise of
a boundary: the oracle reports, per row, how close top_p came to the mass-before of a token at the cut and how
close the uniform number came to an edge of the drawn token's interval.  fp32 sums over a row carry a relative
error of a few 1e-7, so rows with a margin under MARGIN are not compared (and must stay a small minority)."""
import numpy as np
import pytest
import torch

from oracle import ref_sampler as rs
from parrotserve_amd import kernels

pytestmark = pytest.mark.gpu
MARGIN = 5e-6

DT = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def _case(seed, B, V, dtype, std=4.0, quantum=None):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(B, V, generator=g) * std
    if quantum:
        x = torch.round(x / quantum) * quantum  # many equal values
    x = x.to(DT[dtype])
    temps = torch.tensor([1.0, 0.7, 1.3, 0.25])[torch.randint(0, 4, (B,), generator=g)]
    tops = torch.tensor([1.0, 0.95, 0.9, 0.5, 0.1, 1e-6])[torch.randint(0, 6, (B,), generator=g)]
    u = torch.rand(B, generator=g)
    return x, temps, tops, u


def _check(x, temps, tops, u, dtype, min_compared=0.9, stride_pad=0):
    B, V = x.shape
    dev = torch.device("cuda:0")
    if stride_pad:
        buf = torch.full((B, V + stride_pad), 100.0, dtype=x.dtype, device=dev)  # a read past the row would win
        buf[:, :V] = x.to(dev)
        xd = buf[:, :V]
    else:
        xd = x.to(dev)
    ids = kernels.sample_top_p(xd, None if temps is None else temps.to(dev), None if tops is None else tops.to(dev),
                               u.to(dev)).cpu().numpy()
    want, margins = rs.ref_sample(x.double().numpy(), None if temps is None else temps.numpy(),
                                  None if tops is None else tops.numpy(), u.numpy(), dtype)
    assert ids.dtype == np.int64 and ((ids >= 0) & (ids < V)).all()
    clear = margins >= MARGIN
    assert clear.mean() >= min_compared, f"only {clear.sum()} of {B} rows are clear of a boundary"
    bad = np.nonzero(clear & (ids != want))[0]
    assert bad.size == 0, f"rows {bad[:8].tolist()}: got {ids[bad[:8]].tolist()}, want {want[bad[:8]].tolist()}"
    return ids


@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("B,V", [(64, 32000), (3, 1000), (1, 7), (3, 1003), (5, 36864), (4, 50257), (6, 50272),
                                 (3, 57344), (2, 70001)])
def test_matches_oracle(dtype, B, V):
    """Row lengths on every path of the library: rows that fit the register file and start on 16-byte boundaries
    (32000, 1000, 36864, 50272, 57344: the largest), rows that do not start on such boundaries (7, 1003: kept in
    LDS; 50257: re-read) and rows too long for the registers (70001)."""
    x, temps, tops, u = _case(B * 131 + V, B, V, dtype)
    _check(x, temps, tops, u, dtype, min_compared=0.6 if B < 8 else 0.9)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_rows_full_of_equal_values(dtype):
    """Logits on a coarse grid: the cut falls inside a group of equal values, which survive in id order."""
    x, temps, tops, u = _case(5, 48, 4000, dtype, std=2.0, quantum=0.5)
    temps = torch.ones_like(temps)  # a division would spread the grid
    _check(x, temps, tops, u, dtype)


def test_no_filter_no_temperature_and_strided_rows():
    x, _, _, u = _case(9, 32, 32000, "f16")
    a = _check(x, None, None, u, "f16")
    b = _check(x, None, None, u, "f16", stride_pad=24)
    c = _check(x, None, None, u, "f16", stride_pad=3)  # rows off the 16-byte grid: another kernel, same tokens
    assert (a == b).all()
    assert (a == c)[rs.ref_sample(x.double().numpy(), None, None, u.numpy())[1] >= MARGIN].all()


def test_limits_select_the_most_likely_token():
    x, _, _, u = _case(11, 16, 32000, "f16")
    dev = torch.device("cuda:0")
    want = rs.ref_sample(x.double().numpy(), None, np.full(16, 1e-6, dtype=np.float32), u.numpy())[0]
    assert (want == x.double().numpy().argmax(1)).all()
    for temps, tops in [(None, torch.full((16,), 1e-6)), (None, torch.zeros(16)), (torch.zeros(16), None),
                        (torch.full((16,), -1.0), torch.ones(16))]:
        ids = kernels.sample_top_p(x.to(dev), None if temps is None else temps.to(dev),
                                   None if tops is None else tops.to(dev), u.to(dev)).cpu().numpy()
        assert (ids == want).all()


def test_uniform_logits_draw_floor_u_times_v():
    V, B = 64, 512
    g = torch.Generator().manual_seed(3)
    u = torch.rand(B, generator=g)
    dev = torch.device("cuda:0")
    ids = kernels.sample_top_p(torch.zeros(B, V, dtype=torch.float16, device=dev), None, None, u.to(dev)).cpu()
    assert (ids == torch.floor(u * V).long()).all()


def test_masked_tokens_are_never_drawn_and_edges_of_the_range():
    V, B = 1000, 256
    g = torch.Generator().manual_seed(4)
    x = torch.randn(B, V, generator=g).half()
    x[:, ::2] = float("-inf")
    x[0, 1] = 5.0  # certainly inside the filter
    u = torch.rand(B, generator=g)
    u[0], u[1] = 0.0, float(np.nextafter(np.float32(1.0), np.float32(0.0)))
    ids = _check(x, None, torch.full((B,), 0.99), u, "f16")
    assert (ids % 2 == 1).all()
    assert ids[0] == 1  # the first token that can be drawn


def test_draw_frequencies_match_the_probabilities():
    V, B = 16, 65536
    g = torch.Generator().manual_seed(6)
    row = (torch.randn(V, generator=g) * 1.5).half()
    top_p = 0.8
    p, _ = rs.kept_probs(row.double().numpy(), 1.0, top_p, "f16")
    dev = torch.device("cuda:0")
    u = torch.rand(B, generator=torch.Generator(device=dev).manual_seed(1), device=dev)
    ids = kernels.sample_top_p(row.to(dev).expand(B, V).contiguous(), None, torch.full((B,), top_p, device=dev), u)
    counts = torch.bincount(ids.cpu(), minlength=V).numpy()
    assert (counts[p == 0] == 0).all()
    np.testing.assert_allclose(counts / B, p, atol=4 * np.sqrt(0.25 / B))


def test_same_inputs_same_tokens():
    x, temps, tops, u = _case(13, 64, 32000, "bf16")
    dev = torch.device("cuda:0")
    args = (x.to(dev), temps.to(dev), tops.to(dev), u.to(dev))
    a = kernels.sample_top_p(*args)
    b = kernels.sample_top_p(*args)
    assert torch.equal(a, b)


def test_sampler_module_uses_the_kernel():
    """runner.Sampler: top_p -> 0 gives the arg-max of hidden @ W.T; a plain draw stays inside the vocabulary and
    follows torch's generator (same seed, same tokens)."""
    from parrotserve_amd.runner import LlamaConfig, Sampler, SamplingConfig

    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(2)
    W = (torch.randn(4096, 256, generator=g) * 0.05).half().to(dev)
    h = torch.randn(8, 256, generator=g).half().to(dev)
    cfg = LlamaConfig(vocab_size=4096, hidden_size=256)
    s = Sampler(cfg, W)
    ids = s(h, [SamplingConfig(top_p=1e-6)] * 8)
    logits = (h @ W.t()).double().cpu().numpy()
    want = rs.ref_sample(logits, None, np.full(8, 1e-6, dtype=np.float32), np.zeros(8, dtype=np.float32))[0]
    assert ids.cpu().tolist() == want.tolist()
    torch.manual_seed(5)
    a = s(h, [SamplingConfig(temperature=0.8, top_p=0.9)] * 8)
    torch.manual_seed(5)
    b = s(h, [SamplingConfig(temperature=0.8, top_p=0.9)] * 8)
    assert torch.equal(a, b) and int(a.min()) >= 0 and int(a.max()) < 4096
    assert s(h[:0], []).shape == (0,)


@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("B,V", [(16, 32000), (3, 1003), (2, 50257)])
def test_filtered_probabilities_match_oracle(dtype, B, V):
    """ph_top_p_probs: the tensor the reference hands to torch.multinomial (models/sampler.py:58-64) -- soft-max of
    the tokens the top-p filter keeps, zero elsewhere -- against the float64 oracle, on rows whose cut is clear of
    rounding noise: same support, probabilities to fp32 accuracy."""
    x, temps, tops, _ = _case(31 + V, B, V, dtype)
    dev = torch.device("cuda:0")
    probs = kernels.top_p_probs(x.to(dev), temps.to(dev), tops.to(dev)).cpu().double().numpy()
    assert probs.shape == (B, V)
    compared = 0
    for b in range(B):
        want, margin = rs.kept_probs(x[b].double().numpy(), float(temps[b]), float(tops[b]), dtype)
        np.testing.assert_allclose(probs[b].sum(), 1.0, rtol=1e-5)
        if margin < MARGIN:
            continue
        compared += 1
        assert ((probs[b] > 0) == (want > 0)).all(), f"row {b}: support differs"
        np.testing.assert_allclose(probs[b], want, rtol=2e-5, atol=1e-9)
    assert compared >= 0.8 * B


def test_reference_draw_mode_of_the_sampler_module():
    """Sampler.reference_draw: torch.multinomial on the kernel's filtered probabilities -- the reference's own call
    sequence from there on (models/sampler.py:63-64), so for one seed the ids equal torch.multinomial's on the oracle
    path of torch ops (division, sort, cumulative sum, mask, soft-max) whenever the two probability tensors agree."""
    from parrotserve_amd.runner import LlamaConfig, Sampler, SamplingConfig

    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(4)
    W = (torch.randn(4096, 256, generator=g) * 0.3).half().to(dev)  # logits of a few units: a nucleus of tens of tokens
    h = torch.randn(16, 256, generator=g).half().to(dev)
    s = Sampler(LlamaConfig(vocab_size=4096, hidden_size=256), W)
    s.reference_draw = True
    cfgs = [SamplingConfig(temperature=0.8, top_p=0.9)] * 16
    torch.manual_seed(11)
    ids = s(h, cfgs)
    assert ids.shape == (16,) and ids.dtype == torch.int64
    # the reference's sequence of torch calls on the same logits, same seed
    logits = torch.matmul(h, W.t())
    logits.div_(torch.full((16, 1), 0.8, dtype=logits.dtype, device=dev))
    sl, si = logits.sort(dim=-1, descending=True)
    pr = sl.softmax(dim=-1)
    mask = (pr.cumsum(dim=-1) - pr) > torch.full((16, 1), 0.9, dtype=logits.dtype, device=dev)
    sl[mask] = -float("inf")
    logits = torch.gather(sl, dim=-1, index=torch.argsort(si, dim=-1))
    probs = torch.softmax(logits, dim=-1, dtype=torch.float)
    torch.manual_seed(11)
    want = torch.multinomial(probs, num_samples=1, replacement=True).squeeze(-1)
    mine = kernels.top_p_probs(torch.matmul(h, W.t()), torch.full((16,), 0.8, device=dev), torch.full((16,), 0.9, device=dev))
    same_support = ((mine > 0) == (probs > 0)).all(dim=-1)
    # (the torch path rounds its probabilities and their running sums to fp16, which can move a cut by a token)
    assert same_support.float().mean() >= 0.75
    assert torch.equal(ids[same_support], want[same_support])


@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
def test_histogram_cut_on_unusual_rows(dtype):
    """Rows at the edges of the mass histograms: one value everywhere (whole waves on one bin, ranks decide), almost
    everything masked, values that span far more than the histogram's least mass, temperatures outside the range of the
    reciprocal form, a cut between two neighbouring values of the element type."""
    g = torch.Generator().manual_seed(31)
    V = 4000
    rows, temps, tops = [], [], []

    def add(row, temp, top):
        rows.append(row), temps.append(temp), tops.append(top)

    add(torch.zeros(V), 1.0, 0.37013)
    add(torch.full((V,), -3.5), 0.7, 0.90009)
    masked = torch.full((V,), -float("inf"))
    masked[::997] = torch.tensor([1.0, 2.0, 2.0, 0.5, 1.5])
    add(masked, 0.9, 0.8)
    add(torch.randn(V, generator=g) * 60, 1.0, 0.97)
    add(torch.randn(V, generator=g) * 1e-3, 1.0, 0.6)
    add(torch.where(torch.arange(V) % 2 == 0, 8.0, 8.0078125), 1.0, 0.7003)
    add(torch.randn(V, generator=g) * 4, 1.0, 0.9999)
    if dtype != "f16":
        add(torch.randn(V, generator=g) * 1e-13, 2.0 ** -42, 0.9)
        add(torch.randn(V, generator=g) * 1e13, 2.0 ** 42, 0.9)
    x = torch.stack(rows).to(DT[dtype])
    _check(x, torch.tensor(temps), torch.tensor(tops), torch.rand(len(rows), generator=g), dtype, min_compared=0.7)


@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
def test_rows_without_a_finite_mass_take_the_general_rule(dtype):
    """NaN, +inf and nothing but -inf: the same token as from the kernel for rows off the 16-byte grid."""
    g = torch.Generator().manual_seed(32)
    V = 2000
    x = torch.randn(8, V, generator=g) * 3
    x[0, 17] = float("nan")
    x[1, 5] = x[1, 1900] = float("inf")
    x[2] = -float("inf")
    x[3, 11], x[3, 12] = float("nan"), float("inf")
    x[4, 100:] = -float("inf")
    x = x.to(DT[dtype]).cuda()
    temps, tops = torch.tensor([1.0, 0.7] * 4).cuda(), torch.tensor([0.9, 0.5, 1.0, 0.3] * 2).cuda()
    u = torch.rand(8, generator=g).cuda()
    buf = torch.zeros(8, V + 8, dtype=x.dtype, device="cuda")
    buf[:, 1:V + 1] = x
    assert torch.equal(kernels.sample_top_p(x, temps, tops, u), kernels.sample_top_p(buf[:, 1:V + 1], temps, tops, u))


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("value", [1e3, 1e10, 2.3e38, 2.4e38, 3e38, -3e38])
def test_huge_logits_beside_an_infinite_one_take_the_general_rule(dtype, value):
    """A row that holds +inf keeps its logits as they are (no maximum to subtract): the exponential of the largest finite
    ones is +inf, not NaN, and the same token comes out as from the kernel for rows off the 16-byte grid."""
    V = 2000
    x = torch.full((4, V), -200.0)
    x[:, 3], x[:, 1900] = float("inf"), value
    x[1, 5] = float("nan")
    x = x.to(DT[dtype]).cuda()
    buf = torch.zeros(4, V + 8, dtype=x.dtype, device="cuda")
    buf[:, 1:V + 1] = x
    u = torch.tensor([0.5, 0.5, 0.0, 0.9]).cuda()
    for temps, tops in ((None, None), (torch.full((4,), 0.7), torch.tensor([0.9, 0.5, 1.0, 0.3]))):
        args = [t if t is None else t.cuda() for t in (temps, tops)]
        ids = kernels.sample_top_p(x, *args, u)
        assert torch.equal(ids, kernels.sample_top_p(buf[:, 1:V + 1], *args, u))
        assert ids[0] == (1900 if value > 0 else 3)  # no running sum passes an infinite goal: the last token with mass


@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("V", [4000, 32000])
def test_rows_of_few_distinct_values(dtype, V):
    """Rows of 1 to 32 values at random, of a tenth at one value, and nearly flat ones: on both sides of the share of
    equal values from which 16-bit rows are bisected."""
    g = torch.Generator().manual_seed(33)
    rows = [(torch.rand(V, generator=g) * n).floor() * step for n in (1, 2, 3, 4, 5, 6, 8, 16, 32) for step in (0.01, 0.3)]
    rows += [(torch.rand(V, generator=g) < 0.1).float() * 3]
    rows += [torch.randn(V, generator=g) * std for std in (1e-3, 5e-3, 1e-2, 2.5e-2)]
    rows += [(torch.randn(V, generator=g) * 4).clamp(max=0)]
    x = torch.stack(rows).to(DT[dtype])
    tops = torch.tensor([0.9003, 0.3007, 0.6002])[torch.arange(len(rows)) % 3]
    _check(x, torch.ones(len(rows)), tops, torch.rand(len(rows), generator=g), dtype, min_compared=0.6)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_the_time_does_not_hang_on_equal_values(dtype):
    """64 rows of equal logits, of two values and of a value with one other in ten take 1.0 to 1.1 times what normal
    logits take (4.2 to 7.5 times where every such row goes through the histograms): the line is drawn at 2.2."""
    g = torch.Generator(device="cuda").manual_seed(34)
    B, V = 64, 32000
    temps, tops = torch.ones(B, device="cuda"), torch.full((B,), 0.9, device="cuda")
    u = torch.rand(B, generator=g, device="cuda")

    def best(x):
        x = x.to(DT[dtype])
        times = []
        for _ in range(8):
            a, b = torch.cuda.Event(True), torch.cuda.Event(True)
            a.record()
            for _ in range(20):
                kernels.sample_top_p(x, temps, tops, u)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    normal = best(torch.randn(B, V, generator=g, device="cuda") * 4)
    coins = torch.rand(B, V, generator=g, device="cuda")
    for rows in (torch.zeros(B, V, device="cuda"), (coins < 0.5).float() * 0.5, (coins < 0.1).float() * 3):
        assert best(rows) < 2.2 * normal


@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("V", [5, 8191, 8192, 8193, 32761, 32768, 32769, 57337])
def test_row_lengths_around_the_rounds_and_forms_of_the_register_kernel(dtype, V):
    """No whole chunk, a last chunk of one token and of all but one, a round that is full and one that holds a single
    chunk, the longest row of the 32-token form and the shortest of the other; rows start on the 16-byte grid whatever
    their length.  Values in steps of 1/4 (several equal ones at every cut, ranked over rounds and waves), and values so
    close that the finer bin in question holds several, so that its last bits decide (in 32-bit rows: 16-bit rows this
    close are bisected)."""
    B = 6
    pad = -V % 8 + 8
    x, temps, tops, u = _case(V, B, V, dtype, quantum=0.25)
    _check(x, temps, tops, u, dtype, min_compared=0.5, stride_pad=pad)
    g = torch.Generator().manual_seed(V)
    # in steps of 2^-22: fp32 exponentials just under 1 lie 2^-24 apart and are right to one such step, so values closer
    # than 2^-23 may share one, and the kernel ranks equal exponentials by id
    close = ((torch.rand(B, V, generator=g) * 1024).floor() * 2.0 ** -22).to(DT[dtype])
    _check(close, torch.ones(B), torch.tensor([0.9003, 0.3007, 0.6002] * 2), u, dtype, min_compared=0.3, stride_pad=pad)


def _histogram_levels(x, p, chunk):
    """What the register kernel's histograms meet on these rows, from fp32 exponentials: the share of equal and of nearly
    equal values it would look at, and how many values the finer bin holds that the mass crosses `p` in."""
    out = []
    for row, top in zip(x.float().numpy(), p.numpy()):
        first = row[::chunk][: len(row) // chunk // 64 * 64].reshape(-1, 64)
        share = ((np.abs(first - first[:, :1]) < 0.011).sum() + 2 * (first == first[:, :1]).sum()) / first.size
        e = np.sort(np.exp(row - row.max()))[::-1]
        at = np.searchsorted(np.cumsum(e, dtype=np.float64), top * e.sum(dtype=np.float64))
        bins = e.view(np.uint32) >> 10
        out.append((share, len(np.unique(e[bins == bins[min(at, len(e) - 1)]]))))
    return out


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("V", [8191, 32000, 32769])
def test_last_bits_of_the_cut_in_16_bit_rows(dtype, V):
    """16-bit rows that go through the histograms and whose cut falls among values so close that the finer bin holds
    several: the first token of every 16-byte chunk, which is where the kernel looks for few distinct values, spreads over
    31 units, the others lie in steps of 2^-22 (fp16) and 2^-20 (bf16) one unit below the maximum."""
    B, step = 6, 2.0 ** (-22 if dtype == "f16" else -20)
    g = torch.Generator().manual_seed(V)
    x = (torch.rand(B, V, generator=g) * 128).floor() * step
    x[:, ::8] = torch.rand(B, x[:, ::8].shape[1], generator=g) * 31 - 30
    x[:, 0] = 1.0
    x = x.to(DT[dtype])
    tops = torch.tensor([0.9003, 0.3007, 0.6002] * 2)
    for share, values in _histogram_levels(x, tops, 8):
        assert share < 0.5 and values > 1
    _check(x, torch.ones(B), tops, torch.rand(B, generator=g), dtype, min_compared=0.3, stride_pad=-V % 8 + 8)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("at", [0.0, 1e-3, 0.9, 50.0, -300.0, 2000.0, 6e4])
def test_rows_bisected_between_the_values_two_looks_leave(dtype, at):
    """16-bit rows of so few distinct values, or so close ones, that their cut is bisected, and of more than the two looks
    at halfway cuts resolve: neighbouring values of the type around small, large and negative logits (subnormal
    exponentials among them), and nearly flat rows across zero."""
    V, B = 4000, 12
    g = torch.Generator().manual_seed(int(abs(at)) + 41)
    top = torch.tensor(at).to(DT[dtype])
    bits = top.view(torch.int16).to(torch.int32)
    steps = (torch.rand(B // 2, V, generator=g) * torch.tensor([4.0, 5.0, 4.0, 5.0, 4.0, 5.0])[:, None]).floor()
    near = (bits - steps if at >= 0 else bits + steps).to(torch.int16).view(DT[dtype]).float()
    if at == 0.0:
        near = steps * -(2.0 ** -10)
    x = torch.cat([near, at + torch.randn(B // 2, V, generator=g) * 4e-3]).to(DT[dtype])
    tops = torch.tensor([0.9003, 0.3007, 0.6002, 0.9701])[torch.arange(B) % 4]
    temps = torch.tensor([1.0, 1.0, 0.7 if at < 6e4 else 1.0])[torch.arange(B) % 3]
    _check(x, temps, tops, torch.rand(B, generator=g), dtype, min_compared=0.5)
