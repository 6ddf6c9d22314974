"""Path sums written out (taylor_tree) and looked up (addIncoherentPower) at the shapes where their
kernels change: tile edges, odd widths, one or several 256-row time blocks, each sample type. Float
additions are in the reference's order, so the bar is equality with the oracle."""

import numpy as np
import pytest

import seticore_amd as sc

pytestmark = pytest.mark.gpu


def _data(T, N, dtype, seed):
    import torch
    x = torch.from_numpy(np.random.default_rng(seed).exponential(size=(T, N)).astype(np.float32))
    code, kind = {"f32": (sc.SC_F32, torch.float32), "f16": (sc.SC_F16, torch.float16),
                  "bf16": (sc.SC_BF16, torch.bfloat16)}[dtype]
    x = x.to(kind)
    return x.float().numpy(), x.cuda(), code


def _valid(T, N, b):
    last = np.arange(N)[None, :] + (T - 1) * b + np.arange(T)[:, None]
    return (last >= 0) & (last < N)


# Tile widths: 240 channels at 16 rows, 224 / 192 / 184 / 180 at 32 / 64 / 128 / 256.
@pytest.mark.parametrize("T,N,dtype", [
    (2, 4097, "f32"), (16, 239, "f16"), (16, 1201, "bf16"), (32, 225, "f32"), (64, 192, "bf16"),
    (64, 1155, "f32"), (128, 183, "f32"), (128, 1471, "f16"), (256, 181, "f32"),
    (256, 1441, "bf16"), (512, 2003, "f32"), (1024, 4001, "f16")])
def test_tree_at_tile_edges(gpu, oracle, T, N, dtype):
    host, x, code = _data(T, N, dtype, T + N)
    dd = sc.Dedopplerer(T, N, 1.0, 1.0)
    for b in (-1, 0, 1):
        print("tree", T, N, dtype, b, flush=True)
        got = dd.taylor_tree(sc.FilterbankBuffer(T, N, data=x, dtype=code), b).cpu().numpy()
        ok = _valid(T, N, b)
        np.testing.assert_array_equal(got[ok], oracle.basic_taylor_tree(host, b)[ok])


# Levels above 256 run in memory, four channels per thread and 1024 per workgroup.
@pytest.mark.parametrize("T,N", [(512, 513), (512, 1024), (512, 1027), (1024, 2050), (2048, 4099)])
def test_tree_levels_in_memory(gpu, oracle, T, N):
    host, x, code = _data(T, N, "f32", T + N)
    dd = sc.Dedopplerer(T, N, 1.0, 1.0)
    for b in (-1, 0, 1):
        print("levels", T, N, b, flush=True)
        got = dd.taylor_tree(sc.FilterbankBuffer(T, N, data=x, dtype=code), b).cpu().numpy()
        ok = _valid(T, N, b)
        np.testing.assert_array_equal(got[ok], oracle.basic_taylor_tree(host, b)[ok])


# Above 256 rows the path maxima are taken from memory, 32 offsets of four channels per thread; ties
# between offsets and drift blocks keep the reference's first.
@pytest.mark.parametrize("T,N,ties", [(300, 1024, False), (512, 1027, True), (600, 5001, True),
                                      (2048, 515, False)])
def test_search_above_256_rows(gpu, oracle, T, N, ties):
    T_r = sc.round_up_to_power_of_two(T)
    host = np.zeros((T_r, N), np.float32)
    host[:T] = np.random.default_rng(T).exponential(size=(T, N))
    if ties:
        host = np.rint(host)
    foff, tsamp = -2.79e-6, 18.25
    max_drift = 2.6 * abs(1e6 * foff) / tsamp
    import torch
    dd = sc.Dedopplerer(T, N, foff, tsamp)
    hits = []
    print("search", T, N, ties, flush=True)
    dd.search(sc.FilterbankBuffer(T_r, N, data=torch.from_numpy(host).cuda()),
              sc.FilterbankMetadata(coarse_channel_size=N), sc.NO_BEAM, 0, max_drift, 0.0, 2.0, hits)
    ref = oracle.search(host, T, foff, tsamp, max_drift, 0.0, 2.0)
    st = dd.state()
    np.testing.assert_array_equal(st["top_sums"], ref.top_sums)
    pos = ref.top_sums > 0
    np.testing.assert_array_equal(st["top_blocks"][pos], ref.top_blocks[pos])
    np.testing.assert_array_equal(st["top_offsets"][pos], ref.top_offsets[pos])
    assert [(h.index, h.drift_steps) for h in hits] == [(h["index"], h["drift_steps"]) for h in ref.hits]


def test_tree_output_may_be_the_input(gpu, oracle):
    import ctypes
    T, N = 64, 777
    host, x, code = _data(T, N, "f32", 3)
    dd = sc.Dedopplerer(T, N, 1.0, 1.0)
    sc.check(sc.lib().sc_dd_taylor_tree(dd._h, ctypes.c_void_p(x.data_ptr()), code, T, N, N, 1,
                                        ctypes.c_void_p(x.data_ptr()), None))
    ok = _valid(T, N, 1)
    np.testing.assert_array_equal(x.cpu().numpy()[ok], oracle.basic_taylor_tree(host, 1)[ok])


@pytest.mark.parametrize("T,N,dtype,n", [(2, 500, "f32", 1), (16, 9001, "bf16", 257),
                                         (50, 3000, "f16", 40), (64, 3000, "f32", 33),
                                         (128, 4000, "f32", 20), (512, 6000, "f32", 12)])
def test_incoherent_power_of_any_path(gpu, oracle, T, N, dtype, n):
    T_r = sc.round_up_to_power_of_two(T)
    host, x, code = _data(T_r, N, dtype, T)
    dd = sc.Dedopplerer(T, N, 1.0, 1.0)
    rng = np.random.default_rng(n)
    span = T_r - 1
    hits = []
    for d in rng.choice(np.arange(-3 * span, 3 * span + 1), size=min(n, 6 * span + 1), replace=False):
        c = int(rng.integers(max(0, -d), N - max(0, d)))
        hits.append(sc.DedopplerHit(index=c, drift_steps=int(d)))
    print("incoherent", T, N, dtype, len(hits), flush=True)
    dd.addIncoherentPower(sc.FilterbankBuffer(T_r, N, data=x, dtype=code), hits)
    trees = {}
    for h in hits:
        b, p = divmod(h.drift_steps, span)
        if b not in trees:
            trees[b] = oracle.basic_taylor_tree(host, b)
        assert h.incoherent_power == trees[b][p, h.index]
    assert [h.drift_steps for h in hits] == sorted(h.drift_steps for h in hits)


# The output holds the intermediates where it is large enough (16 rows: from about 2 300 channels on in
# 16 bits) and apart from the input; odd widths, more rows than a load group, strided rows.
@pytest.mark.parametrize("T,N,stride,dtype", [
    (1, 1, 1, "f32"), (16, 1000, 1000, "bf16"), (16, 2401, 2403, "f16"), (17, 5003, 5003, "bf16"),
    (13, 70001, 70001, "f32"), (100, 4099, 4100, "bf16")])
def test_normalize_against_float64(gpu, T, N, stride, dtype):
    import torch
    code, kind = {"f32": (sc.SC_F32, torch.float32), "f16": (sc.SC_F16, torch.float16),
                  "bf16": (sc.SC_BF16, torch.bfloat16)}[dtype]
    rng = np.random.default_rng(N)
    x = (rng.exponential(size=(T, stride)) * 3.0 + 1000.0).astype(np.float32)
    if N > 1000:
        x[:, N // 3] = 1e8  # an interferer that holds nearly all of the power
    d = torch.from_numpy(x).cuda()[:, :N]
    print("normalize", T, N, stride, dtype, flush=True)
    y, loc, sd = sc.normalize(d, code)
    colsum = np.zeros(N, np.float32)
    for t in range(T):
        colsum += x[t, :N]
    assert loc == float(np.partition(colsum, N // 2)[N // 2]) / T
    v = x[:, :N].astype(np.float64)
    # A few hundred FP64 roundings at most separate the merged moments from the two-pass ones.
    np.testing.assert_allclose(sd, v.std(), rtol=1e-12, atol=0)
    div = np.float32(sd if sd > 0 else 1.0)
    want = ((v - loc).astype(np.float32) / div).clip(-65504.0, 65504.0)
    np.testing.assert_array_equal(y.cpu().float().numpy(),
                                  torch.from_numpy(want).to(kind).float().numpy())
    if dtype == "f32" and stride == N:
        z, loc2, sd2 = sc.normalize(d, code, out=d)  # in place
        assert (loc2, sd2) == (loc, sd)
        np.testing.assert_array_equal(z.cpu().numpy(), y.cpu().numpy())


def test_normalize_from_several_threads(gpu):
    import torch
    from concurrent.futures import ThreadPoolExecutor
    x = [torch.from_numpy(np.random.default_rng(i).exponential(size=(16, 20001)).astype(np.float32) * (i + 1)).cuda()
         for i in range(8)]
    want = [sc.normalize(v, sc.SC_BF16) for v in x]
    torch.cuda.synchronize()

    def many(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            return [sc.normalize(x[i], sc.SC_BF16) for _ in range(5)]

    print("normalize, 8 threads", flush=True)
    with ThreadPoolExecutor(8) as pool:
        for i, got in enumerate(pool.map(many, range(8))):
            for y, loc, sd in got:
                assert (loc, sd) == want[i][1:]
                assert torch.equal(y, want[i][0])


# An output in pinned host memory takes no intermediates (they are read back and added to atomically).
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_normalize_into_host_memory(gpu, dtype):
    import torch
    T, N = 16, 70001
    code, kind = {"f32": (sc.SC_F32, torch.float32), "bf16": (sc.SC_BF16, torch.bfloat16)}[dtype]
    _, x, _ = _data(T, N, "f32", 8)
    want, loc, sd = sc.normalize(x, code)
    out = torch.empty((T, N), dtype=kind, pin_memory=True)
    print("normalize to the host", dtype, flush=True)
    got = sc.normalize(x, code, out=out)
    assert got[1:] == (loc, sd)
    assert torch.equal(out, want.cpu())


# Up to 8192 hits are read and written in host memory, more at up to 64 rows copied; one handle, its
# buffers growing and then larger than needed.
@pytest.mark.parametrize("T,dtype", [(2, "f16"), (64, "f32"), (128, "f32")])
def test_incoherent_power_of_many_hits(gpu, oracle, T, dtype):
    N = 3001
    host, x, code = _data(T, N, dtype, T)
    dd = sc.Dedopplerer(T, N, 1.0, 1.0)
    trees = {b: oracle.basic_taylor_tree(host, b) for b in (-1, 0, 1)}
    rng = np.random.default_rng(T)
    for n in (8192, 8193, 20000, 9000):
        d = rng.integers(-(T - 1), 2 * (T - 1), size=n)
        c = rng.integers(np.maximum(0, -d), N - np.maximum(0, d))
        hits = [sc.DedopplerHit(index=int(i), drift_steps=int(s)) for i, s in zip(c, d)]
        print("many hits", T, dtype, n, flush=True)
        dd.addIncoherentPower(sc.FilterbankBuffer(T, N, data=x, dtype=code), hits)
        steps = np.array([h.drift_steps for h in hits])
        index = np.array([h.index for h in hits])
        got = np.array([h.incoherent_power for h in hits], np.float32)
        block, offset = np.divmod(steps, T - 1)
        want = np.empty(n, np.float32)
        for b in trees:
            m = block == b
            want[m] = trees[b][offset[m], index[m]]
        np.testing.assert_array_equal(got, want)


# Path sums into pinned host memory: written there up to 512 rows, copied above.
@pytest.mark.parametrize("T", [16, 64, 512, 1024])
def test_tree_into_host_memory(gpu, T):
    import ctypes
    import torch
    N = 2003
    _, x, code = _data(T, N, "f32", T)
    dd = sc.Dedopplerer(T, N, 1.0, 1.0)
    want = dd.taylor_tree(sc.FilterbankBuffer(T, N, data=x, dtype=code), 1).cpu().numpy()
    out = torch.zeros((T, N), pin_memory=True)
    print("tree to the host", T, flush=True)
    sc.check(sc.lib().sc_dd_taylor_tree(dd._h, ctypes.c_void_p(x.data_ptr()), code, T, N, N, 1,
                                        ctypes.c_void_p(out.data_ptr()), None))
    ok = _valid(T, N, 1)
    np.testing.assert_array_equal(out.numpy()[ok], want[ok])
