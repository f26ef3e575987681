"""Time loops whose steps swap two arrays in LDS, compiled once for odd and once for even steps: reads that end in the first,
the second and the odd step out, against the float64 oracle and the loop that is not taken apart; loops inside each other."""
import re

import numpy as np
import pytest

import oracle
import parpy_amd as parpy
from parpy_amd import workloads as W
from parpy_amd.compile import hiprtc_compile

torch = pytest.importorskip("torch")


def opts(n, threads, **kw):
    o = parpy.par({'inst': parpy.threads(n), 'state': parpy.threads(threads)})
    for name, value in kw.items():
        setattr(o, name, value)
    return o


def text(k, threads, **kw):
    hmm, seqs = W.synthetic_hmm(k, n_inst=4, min_len=10, max_len=30)
    a = np.zeros((4, hmm["num_states"]), dtype=np.float32)
    o = opts(4, threads, **kw)
    return parpy.print_compiled(W.forward_syn, [hmm, seqs, np.zeros(4, dtype=np.float32), a, a.copy()], o)


def test_one_text_for_both_parities():
    s = text(5, 1024)
    assert s.count("const auto parpy_step = [&](auto parpy_odd, const int t_") == 1 and s.count("if (parpy_odd.value) {") == 1
    assert "parpy_step(parpy_flag<true>()" in s and "parpy_step(parpy_flag<false>()" in s
    assert "parpy_step" not in text(5, 1024, opt_pair_steps=False)
    assert "parpy_step" not in text(7, 1024)      # the registers of a thread are taken by its tables


@pytest.mark.parametrize("k,taken", [(3, False), (4, True)])
def test_a_step_under_a_test_needs_several_elements_per_thread(k, taken):
    hmm, seqs = W.random_reference_model(k, n_reads=2, min_len=3, max_len=6)
    a = np.zeros((2, hmm["num_states"]), np.float32)
    s = parpy.print_compiled(W.forward_kernel, [hmm, seqs, a, a.copy(), np.zeros(2, np.float32)], opts(2, 1024))
    assert ("parpy_step" in s) == taken


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["reference", "grouped", "scaled"])
@pytest.mark.parametrize("k,threads", [(3, 64), (4, 64), (5, 256)])
def test_reads_of_odd_and_even_length(k, threads, form):
    n = 12
    hmm, seqs = W.synthetic_hmm(k, n_inst=n, min_len=20, max_len=41)
    seqs["lens"][:6] = [1, 2, 3, 4, 5, 6]
    got = {}
    for pairs in (True, False):
        hd, sd = W.to_device(hmm), W.to_device(seqs)
        if form != "reference":
            hd = W.scaled_tables_on_device(hd)
        a1 = torch.zeros((n, hmm["num_states"]), dtype=torch.float32, device="cuda")
        a2 = torch.zeros_like(a1)
        res = torch.zeros(n, dtype=torch.float64 if form == "scaled" else torch.float32, device="cuda")
        f = {"reference": W.forward_syn, "grouped": W.forward_syn4, "scaled": W.forward_scaled}[form]
        f(hd, sd, res, a1, a2, opts=opts(n, threads, opt_pair_steps=pairs))
        got[pairs] = [x.double().cpu().numpy() for x in (res, a1, a2)]
    want = oracle.hmm_syn_forward(hmm, seqs, np.float64)
    # 41 steps of half a unit in the last place of scores up to 256 (single precision); the scaled form keeps 1e-4
    assert np.abs(got[True][0] - want).max() < (1e-4 if form == "scaled" else 41 * 2.0 ** -16)
    for with_pairs, without in zip(got[True], got[False]):
        np.testing.assert_allclose(with_pairs, without, rtol=1e-5, atol=1e-5 if form != "scaled" else 1e-30)


@parpy.jit
def loops_inside_each_other(a, b, out, N, M, U, T):
    parpy.label('inst')
    for i in range(N):
        for u in range(1, U):
            s = b
            d = a
            if u & 1:
                s = a
                d = b
            parpy.label('state')
            for j in range(M):
                d[i, j] = s[i, (j + 1) % M] * 0.5
            for t in range(u % 2, T):
                s2 = b
                d2 = a
                if t & 1:
                    s2 = a
                    d2 = b
                parpy.label('state')
                for j in range(M):
                    d2[i, j] = s2[i, (j + 1) % M] * (1.0 if u % 2 == 0 else 0.25) + s2[i, j] * (1.0 if u & 1 else 2.0)
            for t in range(1, T):
                s3 = b
                d3 = a
                if t & 1:
                    s3 = a
                    d3 = b
                parpy.label('state')
                for j in range(M):
                    d3[i, j] = s3[i, (j + 2) % M] * (0.5 if u & 1 else 0.25)
        parpy.label('state')
        for j in range(M):
            out[i, j] = a[i, j] - b[i, j]


def test_of_loops_inside_each_other_the_inner_one():
    a = np.zeros((4, 512), np.float32)
    s = parpy.print_compiled(loops_inside_each_other, [a, a.copy(), a.copy(), 4, 512, 6, 7], opts(4, 256))
    hiprtc_compile(s[:s.index("// host side")], opts(4, 256))
    step = re.findall(r"const auto parpy_step = \[&\]\(auto parpy_odd, const \w+ (\w+)_\d+\)", s)
    assert step and set(step) == {"t"}
    assert len(re.findall(r"\(u_\d+ & 1\) \? ", s)) == 2 and not re.search(r"parpy_odd\.value\)* \?", s)


@pytest.mark.gpu
@pytest.mark.parametrize("U,T", [(2, 2), (5, 4), (6, 7)])
def test_loops_inside_each_other(U, T):
    n, m = 3, 512
    rng = np.random.default_rng(U)
    a, b = rng.random((n, m)).astype(np.float32), rng.random((n, m)).astype(np.float32)
    out = np.zeros_like(a)
    x, y = a.astype(np.float64), b.astype(np.float64)
    loops_inside_each_other(a, b, out, n, m, U, T, opts=opts(n, 256))
    for u in range(1, U):
        (y if u & 1 else x)[:] = np.roll(x if u & 1 else y, -1, axis=1) * 0.5
        for t in range(u % 2, T):
            s = x if t & 1 else y
            (y if t & 1 else x)[:] = np.roll(s, -1, axis=1) * (1.0 if u % 2 == 0 else 0.25) + s * (1.0 if u & 1 else 2.0)
        for t in range(1, T):
            (y if t & 1 else x)[:] = np.roll(x if t & 1 else y, -2, axis=1) * (0.5 if u & 1 else 0.25)
    # every value is a sum of positive terms of at most 2 * U * T steps, each rounded once to 24 bits
    for got, want in ((a, x), (b, y)):
        np.testing.assert_allclose(got, want, rtol=2 * U * T * 2.0 ** -24)
    assert np.array_equal(out, a - b)


@parpy.jit
def parity_as_a_number(a, b, N, M, T):
    parpy.label('inst')
    for i in range(N):
        for t in range(1, T):
            s = b
            d = a
            if t & 1:
                s = a
                d = b
            parpy.label('state')
            for j in range(M):
                d[i, j] = s[i, (j + 1) % M] + ((t & 1) << 40) - parpy.operators.max(t & 1, j) + (1 if (t & 1) == 0 else 3) + (5 if (t & 1) != 1 and j > 3 else 7) + (~(t & 1)) * (t & 1)


def test_the_parity_as_a_number_keeps_its_width():
    """A shift of a truth value is one of 32 bits."""
    a = np.zeros((4, 512), np.int64)
    s = parpy.print_compiled(parity_as_a_number, [a, a.copy(), 4, 512, 7], opts(4, 256))
    hiprtc_compile(s[:s.index("// host side")], opts(4, 256))
    assert "(int64_t)(t_" in s and "parpy_odd.value <<" not in s
    assert s.count("if (parpy_odd.value) {") == 1 and "(!parpy_odd.value)" in s


@pytest.mark.gpu
@pytest.mark.parametrize("T", [2, 3, 8])
def test_the_parity_as_a_number(T):
    n, m = 3, 512
    rng = np.random.default_rng(T)
    a, b = rng.integers(-1000, 1000, (n, m)), rng.integers(-1000, 1000, (n, m))
    x, y = a.copy(), b.copy()
    parity_as_a_number(a, b, n, m, T, opts=opts(n, 256))
    j = np.arange(m)
    for t in range(1, T):
        p = t & 1
        (y if p else x)[:] = np.roll(x if p else y, -1, axis=1) + (p << 40) - np.maximum(p, j) + (1 if p == 0 else 3) + np.where((p != 1) & (j > 3), 5, 7) + ~p * p
    assert np.array_equal(a, x) and np.array_equal(b, y)
