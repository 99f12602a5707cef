"""GPU parity of the EXL3 linear (the shared expert) and the prefill path through the C ABI against the CPU oracle:
unpack bit-exact, rot_in bit-exact, linear outputs within fp32-accumulation tolerance with the split-K counters
left at zero, the route exactly, and prompt_experts.run within 2e-3 * RMS(out) (also deterministic run to run)."""
import numpy as np
import pytest

import oracle as orc
from helpers import assert_close_rms, oracle_routed

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ea():
    from ea_exl3 import device, linear, moe, prompt_experts, synth

    device.init(0)
    return device, linear, moe, prompt_experts, synth


def _case(synth, M, K, N, k2, seed):
    T = synth.trellis(seed, 0, 0, 0, K, N, k2)
    suh = synth.scales(seed + 1, K, 1.0)
    svh = synth.scales(seed + 2, N, 0.02)
    x = synth.activations(seed + 3, M, K, "bf16")
    return T, suh, svh, x


@pytest.mark.parametrize("k2,cb", [(8, 1), (10, 2), (12, 2), (6, 1)])
def test_unpack_bit_exact(ea, k2, cb):
    device, linear, _, _, synth = ea
    K, N = 256, 512
    T = synth.trellis(60, 0, 0, 0, K, N, k2)
    S = linear.strips(T, K, N, k2)
    tw = 4 * k2
    want = orc.dequant_expert(T, K, N, k2, cb)
    dS, dW = device.upload(S), device.zeros((K, N), torch.int16)
    linear.Kernels().unpack_w(device.stream(), dS.data_ptr(), dW.data_ptr(), K, N, k2, cb, 8 * tw, (K // 16) * 8 * tw)
    np.testing.assert_array_equal(device.download(dW), want)


@pytest.mark.parametrize("M,K,N,k2,cb,y_dtype", [
    (1, 6144, 256, 8, 1, 1),     # the shared expert's gate / up at batch 1 (plan: SK 8, WK 4), bf16 out
    (1, 256, 6144, 8, 1, 2),     # its down (SK 1), fp32 out
    (16, 6144, 256, 10, 2, 2),   # 5-bit mul1 (the real checkpoints' shared expert), 16 rows
    (40, 1024, 640, 8, 2, 0),    # five row passes of the tagged form (few blocks), fp16 out
    (128, 512, 384, 6, 1, 2),    # the most rows a call takes
    (128, 6144, 256, 8, 1, 1),   # the shared expert's gate / up on a 128-row window
    (96, 256, 6144, 8, 1, 2),    # its down on a 96-row window
    (4, 6144, 2048, 8, 1, 2),    # config 1's shape at four rows (the small-row kernel: 32-column groups x 8 splits)
    (7, 2048, 512, 6, 1, 0),     # 3 bits, fp16 out, a ragged row count
    (2, 1024, 384, 4, 1, 2),     # 2 bits
    (3, 2048, 512, 12, 2, 2),    # 6-bit mul1 (widths above 10: the kernel for more rows at any row count)
    (5, 1024, 384, 8, 2, 1),     # 4-bit mul1, bf16 out
    (1, 8192, 256, 8, 1, 2),     # SK 16: the tagged finisher polls eight splits
    (3, 8192, 512, 6, 1, 1),     # the same at three rows, 3 bits, bf16 out
])
def test_linear_call(ea, M, K, N, k2, cb, y_dtype):
    device, linear, _, _, synth = ea
    T, suh, svh, x = _case(synth, M, K, N, k2, 61 + M)
    lin = linear.Linear(T, suh, svh, K, N, k2, cb)
    xh_w = orc.exl3_rot_in(x, suh, M, K, bf16=True)
    tw = 4 * k2
    y_w = orc.exl3_linear(xh_w, linear.strips(T, K, N, k2), 8 * tw, (K // 16) * 8 * tw, svh, M, K, N, k2, cb, lin.sk,
                          lin.wk, y_dtype=2)
    sc = linear.Scratch(128, K, lin.sk * 128 * N)
    dx = device.upload(x)
    y = device.zeros((M, N), torch.float32 if y_dtype == 2 else torch.int16)
    for rep in range(2):  # twice: the counters must be back at zero after each call
        linear.call(device.stream(), sc, [lin], dx.data_ptr(), 1, M, [y.data_ptr()], [y_dtype])
        np.testing.assert_array_equal(device.download(sc.xh[0][: M * K].view(torch.int16)).reshape(M, K), xh_w)
        got = device.download(y)
        if y_dtype == 2:
            assert_close_rms(got, y_w, 1e-4, f"linear M={M} rep={rep}")
        else:  # one rounding to fp16 / bf16 of the fp32 result: half an ulp of the format, plus the fp32 slack
            got = got.view(np.float16).astype(np.float32) if y_dtype == 0 else synth.bf16_to_f32(got)
            eps = 2.0 ** -11 if y_dtype == 0 else 2.0 ** -8
            bound = eps * np.abs(y_w) + 1e-4 * np.sqrt(np.mean(y_w.astype(np.float64) ** 2))
            assert np.all(np.abs(got - y_w) <= bound), f"linear M={M}: rounded output off"
        assert int(device.download(lin.counters).sum()) == 0


def test_linear_call_rotated_matches_call(ea):
    """callRotated on the xh a call leaves in the scratch (the small-row kernel reads it instead of rotating) gives
    the call's result bit for bit; fp16 and bf16 inputs."""
    device, linear, _, _, synth = ea
    M, K, N, k2 = 3, 6144, 2048, 8
    T, suh, svh, x = _case(synth, M, K, N, k2, 90)
    lin = linear.Linear(T, suh, svh, K, N, k2, 1)
    sc = linear.Scratch(M, K, lin.sk * M * N)
    for x_dtype in (0, 1):
        xb = synth.activations(91 + x_dtype, M, K, ["f16", "bf16"][x_dtype])
        dx = device.upload(xb)
        y1, y2 = device.zeros((M, N), torch.float32), device.zeros((M, N), torch.float32)
        linear.call(device.stream(), sc, [lin], dx.data_ptr(), x_dtype, M, [y1.data_ptr()], [2])
        np.testing.assert_array_equal(device.download(sc.xh[0][: M * K].view(torch.int16)).reshape(M, K),
                                      orc.exl3_rot_in(xb, suh, M, K, bf16=x_dtype == 1))
        linear.call_rotated(device.stream(), sc, [lin], M, [y2.data_ptr()], [2])
        np.testing.assert_array_equal(device.download(y1), device.download(y2))
        assert int(device.download(lin.counters).sum()) == 0
    assert device.device_status() == 0


def test_linear_three_jobs_one_launch(ea):
    device, linear, _, _, synth = ea
    M, K = 3, 1024
    shapes = [(256, 8), (512, 8), (128, 8)]
    lins, wants, outs = [], [], []
    x = synth.activations(70, M, K, "f16")
    for i, (N, k2) in enumerate(shapes):
        T = synth.trellis(71 + i, 0, 0, 0, K, N, k2)
        suh, svh = synth.scales(72 + i, K, 1.0), synth.scales(73 + i, N, 0.02)
        lin = linear.Linear(T, suh, svh, K, N, k2, 1)
        lins.append(lin)
        xh = orc.exl3_rot_in(x, suh, M, K)
        tw = 4 * k2
        wants.append(orc.exl3_linear(xh, linear.strips(T, K, N, k2), 8 * tw, (K // 16) * 8 * tw, svh, M, K, N, k2,
                                     1, lin.sk, lin.wk))
        outs.append(device.zeros((M, N), torch.float32))
    sc = linear.Scratch(M, K, max(l.sk * M * l.n for l in lins))
    dx = device.upload(x)
    linear.call(device.stream(), sc, lins, dx.data_ptr(), 0, M, [o.data_ptr() for o in outs], [2, 2, 2])
    for o, w, l in zip(outs, wants, lins):
        assert_close_rms(device.download(o), w, 1e-4, "job")
        assert int(device.download(l.counters).sum()) == 0


@pytest.mark.parametrize("M,K,Ns,k2,cb", [
    (4, 2048, (6144,), 8, 1),       # more blocks than CUs on the one-row kernel: from four rows on here
    (8, 6144, (2048,), 8, 1), (9, 1152, (384,), 6, 1), (15, 6144, (256, 256), 10, 2), (16, 384, (128,), 4, 1),
    (17, 640, (8192,), 8, 2),       # one split, the finish in the block, a ragged chunk (five Hadamard blocks)
    (31, 256, (6144,), 12, 2), (33, 2048, (1024, 128), 8, 1), (64, 6144, (256, 256), 10, 2), (65, 1536, (640,), 12, 2),
    (97, 6144, (2048,), 6, 1), (127, 2048, (6144,), 8, 1),
    # rotated rows (the last call below) on the one-row kernel: flags at twelve rows, and tagged passes side by side
    (12, 1792, (768,), 10, 2), (24, 6144, (256, 256), 8, 1), (120, 6144, (128,), 8, 1),
])
@pytest.mark.parametrize("x_dtype", [1, 2])
def test_linear_many_rows(ea, M, K, Ns, k2, cb, x_dtype):
    """The launches that decode each tile once for all rows: the edges of row tiles, chunks and splits, several jobs,
    rotated inside the products (16-bit x, few blocks) or before them (fp32 x). Against the oracle: fp32 sums of K
    products of fp16 in another order, 1e-4 * RMS as for the other forms."""
    device, linear, _, _, synth = ea
    x = synth.activations(170 + M, M, K, "bf16" if x_dtype == 1 else "f32")
    lins, wants, outs = [], [], []
    for i, N in enumerate(Ns):
        T = synth.trellis(171 + i, 0, 0, 0, K, N, k2)
        suh, svh = synth.scales(172 + i, K, 1.0), synth.scales(173 + i, N, 0.02)
        lin = linear.Linear(T, suh, svh, K, N, k2, cb)
        xh = orc.exl3_rot_in(x, suh, M, K, bf16=x_dtype == 1)
        tw = 4 * k2
        lins.append(lin)
        wants.append((xh, orc.exl3_linear(xh, linear.strips(T, K, N, k2), 8 * tw, (K // 16) * 8 * tw, svh, M, K, N, k2,
                                          cb, lin.sk, lin.wk)))
        outs.append(device.zeros((M, N), torch.float32))
    sc = linear.Scratch(M, K, max(l.sk * M * l.n for l in lins))
    dx = device.upload(x)
    for rep in range(2):
        linear.call(device.stream(), sc, lins, dx.data_ptr(), x_dtype, M, [o.data_ptr() for o in outs], [2] * len(lins))
        for i, (o, (xh, w), l) in enumerate(zip(outs, wants, lins)):
            np.testing.assert_array_equal(device.download(sc.xh[i][: M * K].view(torch.int16)).reshape(M, K), xh)
            assert_close_rms(device.download(o), w, 1e-4, f"M={M} job {i} rep={rep}")
            assert int(device.download(l.counters).sum()) == 0
    first = [device.download(o) for o in outs]
    linear.call_rotated(device.stream(), sc, lins, M, [o.data_ptr() for o in outs], [2] * len(lins))
    for o, w in zip(outs, wants):
        assert_close_rms(device.download(o), w[1], 1e-4, f"M={M} rotated")
    assert device.device_status() == 0 and all(np.isfinite(f).all() for f in first)


@pytest.mark.parametrize("M,K,N,jobs", [(1, 512, 512, 1), (20, 512, 512, 2), (128, 896, 896, 1), (70, 768, 256, 2),
                                        (33, 256, 1024, 1)])
def test_linear_output_in_place_of_the_input(ea, M, K, N, jobs):
    """One K split: the first output takes the input's place (from its first byte on, shorter or longer than it), and the
    rotated rows are taken before any of it is stored: every output's bits are those of a call that leaves x alone."""
    device, linear, _, _, synth = ea
    lins = []
    for i in range(jobs):
        T = synth.trellis(190 + i, 0, 0, 0, K, N, 8)
        lins.append(linear.Linear(T, synth.scales(191 + i, K, 1.0), synth.scales(192 + i, N, 0.02), K, N, 8, 1))
        assert lins[-1].sk == 1
    x = synth.activations(193, M, K, "bf16")
    sc = linear.Scratch(M, K, 1)
    apart, got = [device.zeros((M, N), torch.int16) for _ in lins], [device.zeros((M, N), torch.int16) for _ in lins]
    dx = device.upload(x)
    linear.call(device.stream(), sc, lins, dx.data_ptr(), 1, M, [o.data_ptr() for o in apart], [1] * jobs)
    both = device.zeros((M * max(K, N),), torch.int16)
    both[: M * K] = device.upload(x).view(torch.int16).reshape(-1)
    linear.call(device.stream(), sc, lins, both.data_ptr(), 1, M, [both.data_ptr()] + [o.data_ptr() for o in got[1:]],
                [1] * jobs)
    np.testing.assert_array_equal(device.download(both)[: M * N].reshape(M, N), device.download(apart[0]))
    for a, b in zip(got[1:], apart[1:]):
        np.testing.assert_array_equal(device.download(a), device.download(b))
    # xh in the input's place: the rotation alone writes there
    dx2 = device.upload(x)
    sc.c.xh[0] = dx2.data_ptr()
    y = device.zeros((M, N), torch.int16)
    linear.call(device.stream(), sc, lins[:1], dx2.data_ptr(), 1, M, [y.data_ptr()], [1])
    np.testing.assert_array_equal(device.download(y), device.download(apart[0]))
    assert device.device_status() == 0


def _raw_jobs(specs):
    """ea_exl3_linear's jobs from dicts of Job fields (device addresses and strides in words)."""
    from ea_exl3._lib import Jobs

    jobs = Jobs()
    jobs.n = len(specs)
    for j, spec in zip(jobs.j, specs):
        for name, v in spec.items():
            setattr(j, name, v)
    return jobs


@pytest.mark.parametrize("M", [1, 7, 8, 40])
@pytest.mark.parametrize("K,wk,jobs", [
    (768, 4, ((256, 3, True),)),                                # an odd split count: the flag form below eight rows
    (512, 8, ((128, 2, False), (384, 2, True))),                # eight waves a split: likewise
    (512, 2, ((256, 1, True), (128, 4, True), (384, 1, False))),  # jobs of one split and of several in one call
    (256, 2, ((128, 1, False), (256, 2, True))),
])
def test_linear_bias_and_mixed_splits(ea, M, K, wk, jobs):
    """ea_exl3_linear with a bias, split counts that no plan gives, and jobs of one and of several K splits in one call."""
    device, linear, _, _, synth = ea
    k2, cb = 8, 1
    tw = 4 * k2
    xh = synth.f16_bits(np.random.default_rng(620 + M).standard_normal((M, K)))
    dx = device.upload(xh)
    specs, wants, outs, keep = [], [], [], [dx]
    for i, (N, SK, biased) in enumerate(jobs):
        T = synth.trellis(621 + i, 0, 0, 0, K, N, k2)
        svh = synth.scales(622 + i, N, 0.02)
        bias = synth.scales(623 + i, N, 0.5) if biased else None
        strips = linear.strips(T, K, N, k2)
        wants.append(orc.exl3_linear(xh, strips, 8 * tw, (K // 16) * 8 * tw, svh, M, K, N, k2, cb, SK, wk, bias=bias))
        t, sv, z = device.upload(strips), device.upload(svh), device.zeros(SK * M * N, torch.float32)
        cnt, y = device.zeros(8 * (N // 128), torch.int32), device.zeros((M, N), torch.float32)
        b = device.upload(bias) if biased else None
        keep += [t, sv, z, b, cnt]
        outs.append((y, cnt))
        specs.append(dict(xh=dx.data_ptr(), T=t.data_ptr(), stride_k=8 * tw, stride_nb=(K // 16) * 8 * tw, svh=sv.data_ptr(),
                          bias=b.data_ptr() if biased else 0, y=y.data_ptr(), Z=z.data_ptr() if SK > 1 else 0,
                          counters=cnt.data_ptr(), y_dtype=2, N=N, SK=SK))
    for rep in range(2):
        linear.Kernels().linear(device.stream(), _raw_jobs(specs), M, K, k2, cb, wk)
        for (y, cnt), want in zip(outs, wants):
            assert_close_rms(device.download(y), want, 1e-4, f"M={M} rep {rep}")
            assert int(device.download(cnt).sum()) == 0
            y.fill_(float("nan"))
    assert device.device_status() == 0


@pytest.mark.parametrize("M,SK", [(5, 1), (40, 2)])
@pytest.mark.parametrize("stride", [1 << 27, 1 << 20, -(1 << 20)])
def test_linear_k_strides_of_any_size(ea, M, SK, stride):
    """ea_exl3_linear takes 64-bit tile strides: k tiles half a gigabyte apart (8 GB in all, past 32-bit offsets) and k
    tiles laid out backwards."""
    device, linear, _, _, synth = ea
    K, N, k2, cb = 256, 128, 8, 1
    tw, kt = 4 * k2, K // 16
    T = synth.trellis(600, 0, 0, 0, K, N, k2)
    svh = synth.scales(601, N, 0.02)
    xh = synth.f16_bits(np.random.default_rng(602).standard_normal((M, K)))
    want = orc.exl3_linear(xh, T, 8 * tw, kt * 8 * tw, svh, M, K, N, k2, cb, SK, 2)
    words = torch.empty(kt * abs(stride), dtype=torch.int32, device="cuda")
    first = words.data_ptr() + (0 if stride > 0 else (kt - 1) * -stride * 4)
    tiles = device.upload(T.view(np.int32).reshape(kt, 8 * tw))
    for t in range(kt):
        at = t * stride if stride > 0 else (kt - 1 - t) * -stride
        words[at:at + 8 * tw] = tiles[t]
    dx, dsv = device.upload(xh), device.upload(svh)
    z, cnt = device.zeros(SK * M * N, torch.float32), device.zeros(8 * (N // 128), torch.int32)
    y = device.zeros((M, N), torch.float32)
    jobs = _raw_jobs([dict(xh=dx.data_ptr(), T=first, stride_k=stride, stride_nb=0, svh=dsv.data_ptr(), bias=0,
                           y=y.data_ptr(), Z=z.data_ptr() if SK > 1 else 0, counters=cnt.data_ptr(), y_dtype=2, N=N, SK=SK)])
    linear.Kernels().linear(device.stream(), jobs, M, K, k2, cb, 2)
    assert_close_rms(device.download(y), want, 1e-4, f"k stride {stride}")
    assert device.device_status() == 0


def test_linear_errors(ea):
    device, linear, _, _, synth = ea
    from ea_exl3._lib import EaError

    T, suh, svh, x = _case(synth, 1, 256, 128, 8, 80)
    a = linear.Linear(T, suh, svh, 256, 128, 8, 1)
    T2 = synth.trellis(81, 0, 0, 0, 512, 128, 8)
    b = linear.Linear(T2, synth.scales(82, 512, 1.0), svh, 512, 128, 8, 1)
    sc = linear.Scratch(1, 512, 4096)
    y = device.zeros((1, 128), torch.float32)
    dx = device.upload(x)
    with pytest.raises(EaError) as e:  # different K: not groupable (linear.zig:133-138)
        linear.call(device.stream(), sc, [a, b], dx.data_ptr(), 1, 1, [y.data_ptr()] * 2, [2, 2])
    assert e.value.code == 14
    with pytest.raises(EaError) as e:  # 129 rows
        linear.call(device.stream(), sc, [a], dx.data_ptr(), 1, 129, [y.data_ptr()], [2])
    assert e.value.code == 14


# ---- prefill -------------------------------------------------------------------------------------------------------

def _prompt_case(ea, R, E, D, I, k2, seed, x_dtype=1, zipf=True, cb=1, planes=True):
    device, _, moe, pe, synth = ea
    slots = 8
    pick = synth.picks_zipf(seed, R, 1.1, E, slots) if zipf else synth.picks_uniform(seed, R, E, slots)
    wts = synth.routing_weights(seed + 1, R, slots)
    host = synth.HostLayer(seed + 2, experts=E, dims=D, width=I, k2=k2, cb=cb, only=np.unique(pick))
    x = synth.activations(seed + 3, R, D, ["f16", "bf16", "f32"][x_dtype])
    ex = moe.Routed(host)
    assert pe.supported(ex)
    sc = pe.Scratch(ex, R, slots, planes=planes)
    dx, dp, dw = device.upload(x), device.upload(pick), device.upload(wts)
    return host, ex, sc, x, pick, wts, dx, dp, dw


@pytest.mark.parametrize("R,E,D,I,k2", [(130, 64, 512, 256, 8), (300, 256, 1024, 256, "mixed"), (40, 32, 256, 128, 6),
                                        (120, 32, 256, 128, 12), (300, 32, 256, 128, 12), (300, 32, 256, 128, 8),
                                        # widths above 10; Zipf over 32 experts gives the top experts ~300 pairs: four
                                        # items of up to 80
                                        (300, 32, 256, 128, 11), (300, 32, 256, 128, 14), (300, 32, 256, 128, 16),
                                        (260, 32, 512, 256, "wide-mixed")])
def test_prompt_experts_run(ea, R, E, D, I, k2):
    device, _, _, pe, synth = ea
    if k2 == "wide-mixed":  # two and three trellis words a lane in one layer
        k2v = np.array([(12, 8, 6, 16, 10, 11, 4, 14)[e % 8] for e in range(E)], np.int32)
    else:
        k2v = synth.mixed_widths(5, E) if k2 == "mixed" else k2
    host, ex, sc, x, pick, wts, dx, dp, dw = _prompt_case(ea, R, E, D, I, k2v, 100 + R)
    want = orc.prompt_experts(x, pick, wts, oracle_routed(host), R, 8, bf16=True)
    out = device.zeros((R, D), torch.float32)
    pe.run(device.stream(), dx.data_ptr(), D, dp.data_ptr(), dw.data_ptr(), ex, sc, out.data_ptr(), R, do_round=False)
    got = device.download(out)
    assert_close_rms(got, want, 2e-3, "prompt experts")
    # the same bits on a second run (slots added in order, no atomics in the sums)
    out2 = device.zeros((R, D), torch.float32)
    pe.run(device.stream(), dx.data_ptr(), D, dp.data_ptr(), dw.data_ptr(), ex, sc, out2.data_ptr(), R, do_round=False)
    np.testing.assert_array_equal(device.download(out2), got)
    # do_round: each value through bf16
    pe.run(device.stream(), dx.data_ptr(), D, dp.data_ptr(), dw.data_ptr(), ex, sc, out2.data_ptr(), R, do_round=True)
    np.testing.assert_array_equal(device.download(out2), synth.bf16_to_f32(synth.bf16_bits(got)))
    assert device.device_status() == 0


@pytest.mark.parametrize("planes", [True, False])
def test_prompt_experts_full_shape_512(ea, planes):
    """BASELINE config 4 at its real shape: 512 rows, D 6144, I 256, 256 experts, Zipf(1.1), 4 bits, fp16 x; with the
    pair plane and without it."""
    device, _, _, pe, synth = ea
    R, D = 512, 6144
    host, ex, sc, x, pick, wts, dx, dp, dw = _prompt_case(ea, R, 256, D, 256, 8, 200, x_dtype=0, planes=planes)
    want = orc.prompt_experts(x, pick, wts, oracle_routed(host), R, 8)
    out = device.zeros((R, D), torch.float32)
    pe.run(device.stream(), dx.data_ptr(), D, dp.data_ptr(), dw.data_ptr(), ex, sc, out.data_ptr(), R,
           do_round=False, x_dtype=0)
    assert_close_rms(device.download(out), want, 2e-3, "prompt experts R=512")


@pytest.mark.parametrize("k2", [2, 3, 4, 5, 7, 9, 10])
def test_prompt_experts_every_staged_width(ea, k2):
    """The staged item GEMMs' widths the tests above leave out (K2 6 and 8 are theirs), through both item lists (Zipf
    over 32 experts at 160 rows gives items of both sizes), with the pair plane."""
    device, _, _, pe, synth = ea
    R, E, D, I = 160, 32, 512, 256
    host, ex, sc, x, pick, wts, dx, dp, dw = _prompt_case(ea, R, E, D, I, k2, 900 + k2)
    want = orc.prompt_experts(x, pick, wts, oracle_routed(host), R, 8, bf16=True)
    out = device.zeros((R, D), torch.float32)
    pe.run(device.stream(), dx.data_ptr(), D, dp.data_ptr(), dw.data_ptr(), ex, sc, out.data_ptr(), R, do_round=False)
    assert_close_rms(device.download(out), want, 2e-3, f"prompt experts, K2 {k2}")
    assert device.device_status() == 0


@pytest.mark.parametrize("planes", [True, False])
@pytest.mark.parametrize("k2,R,E", [(2, 20, 64), (3, 20, 64), (5, 20, 64), (3, 100, 24)])
def test_prompt_experts_narrow_widths_resident_down(ea, k2, R, E, planes):
    """Widths whose staged chunk does not fill a wave's 16-byte loads, at a D the resident-activation down kernel takes
    (16 column blocks): lanes that store nothing read the words of lanes that do. Items of at most 6 pairs, and (24
    experts, 100 rows) both lists."""
    device, _, _, pe, synth = ea
    D = 2048
    host, ex, sc, x, pick, wts, dx, dp, dw = _prompt_case(ea, R, E, D, 256, k2, 950 + k2, zipf=False, planes=planes)
    want = orc.prompt_experts(x, pick, wts, oracle_routed(host), R, 8, bf16=True)
    out = device.zeros((R, D), torch.float32)
    pe.run(device.stream(), dx.data_ptr(), D, dp.data_ptr(), dw.data_ptr(), ex, sc, out.data_ptr(), R, do_round=False)
    assert_close_rms(device.download(out), want, 2e-3, f"narrow widths, K2 {k2}, planes={planes}")
    assert device.device_status() == 0


@pytest.mark.parametrize("k2,cb,R,E,I", [(13, 1, 20, 64, 256), (15, 2, 100, 24, 256), (16, 0, 100, 24, 128), (11, 0, 300, 24, 256)])
def test_prompt_experts_wide_widths_resident_down(ea, k2, cb, R, E, I):
    """Widths above 10 (three trellis words a lane) through both item lists and the resident-activation down kernel,
    every codebook; both plane modes give the same bits."""
    device, _, _, pe, synth = ea
    D = 2048
    host, ex, sc, x, pick, wts, dx, dp, dw = _prompt_case(ea, R, E, D, I, k2, 970 + k2, zipf=False, cb=cb)
    want = orc.prompt_experts(x, pick, wts, oracle_routed(host), R, 8, bf16=True)
    got = []
    for planes in (True, False):
        out = device.zeros((R, D), torch.float32)
        pe.run(device.stream(), dx.data_ptr(), D, dp.data_ptr(), dw.data_ptr(), ex, pe.Scratch(ex, R, 8, planes=planes),
               out.data_ptr(), R, do_round=False)
        got.append(device.download(out))
        assert_close_rms(got[-1], want, 2e-3, f"wide widths, K2 {k2}, planes={planes}")
    np.testing.assert_array_equal(got[0], got[1])
    assert device.device_status() == 0


@pytest.mark.parametrize("planes", [True, False])
@pytest.mark.parametrize("R,k2,cb", [(40, 12, 1), (300, 11, 2), (300, 16, 0), (1100, "wide-mixed", 1)])
def test_prompt_experts_wide_layers_sum_k_in_order(ea, R, k2, cb, planes):
    """A layer that holds a width above 10 sums gate and up over all of K in ascending order, in one accumulator. Block 0
    of K (128 columns) puts one large product into every sum and block 2, with block 0's tiles and the opposite sign, takes
    it out again: in that order exactly, so the last block's small products leave the same bits as without the two. Sums of
    K's halves, added at the end, lose the small products' low bits against the large one (2^-24 of 4e4 is 1 % of them)."""
    device, _, moe, pe, synth = ea
    E, D, I = 24, 512, 256
    k2v = np.array([(12, 8, 6, 16, 10, 11, 4, 14)[e % 8] for e in range(E)], np.int32) if k2 == "wide-mixed" else k2
    pick, wts = synth.picks_zipf(810 + R, R, 1.1, E, 8), synth.routing_weights(811, R, 8)
    host = synth.HostLayer(812, experts=E, dims=D, width=I, k2=k2v, cb=cb, only=np.unique(pick))
    for m in (0, 1):
        for t in host.trellis[m]:
            if t is not None:
                rows = t.reshape(D // 16, -1)
                rows[16:24] = rows[0:8]
    host.suh_g = host.suh_u = synth.f16_bits(np.ones(E * D))
    small = np.zeros((R, D), np.float32)
    small[:, 384:] = synth.bf16_to_f32(synth.bf16_bits(0.015 * synth.activations(813, R, D, "f32")[:, 384:]))
    had = np.array([[(-1.0) ** bin(i & j).count("1") for j in range(128)] for i in range(128)], np.float32)
    both = small.copy()
    both[:, 0:128] = 4096.0 * had[np.arange(R) % 128]  # rotated: one entry of 4096 sqrt(128), the others exactly zero
    both[:, 256:384] = -both[:, 0:128]
    ex = moe.Routed(host)
    sc = pe.Scratch(ex, R, 8, planes=planes)
    dp, dw = device.upload(pick), device.upload(wts)
    got = []
    for x in (small, both):
        dx = device.upload(synth.bf16_bits(x))
        out = device.zeros((R, D), torch.float32)
        pe.run(device.stream(), dx.data_ptr(), D, dp.data_ptr(), dw.data_ptr(), ex, sc, out.data_ptr(), R, do_round=False)
        got.append(device.download(out))
    want = orc.prompt_experts(synth.bf16_bits(small), pick, wts, oracle_routed(host), R, 8, bf16=True)
    assert_close_rms(got[0], want, 2e-3, f"wide layer, small rows, K2 {k2}")
    np.testing.assert_array_equal(got[1], got[0])
    assert device.device_status() == 0


@pytest.mark.parametrize("x_dtype,pad,planes", [(0, 0, True), (1, 8, False), (1, 2, False)])
def test_prompt_experts_long_pass_rotations(ea, x_dtype, pad, planes):
    """More than 1,024 rows: the larger items' products rotate x themselves (16-bit rows on 16-byte boundaries, strided or
    not) or, for rows that do not lie so (pad 2), read rotated pairs: the oracle's bar, and a row's bits are those of the
    same row in a shorter pass, which always takes the rotation launch."""
    device, _, moe, pe, synth = ea
    R, E, D, I, short = 1030, 48, 512, 256, 200
    pick, wts = synth.picks_zipf(990, R, 1.1, E, 8), synth.routing_weights(991, R, 8)
    pick[3, 2] = -1  # a slot without an expert
    host = synth.HostLayer(992, experts=E, dims=D, width=I, k2=synth.mixed_widths(5, E), cb=1, only=np.unique(pick[pick >= 0]))
    x = synth.activations(993, R, D, ["f16", "bf16"][x_dtype])
    wide = np.zeros((R, D + pad), np.uint16)
    wide[:, :D] = x
    ex = moe.Routed(host)
    dx, dp, dw = device.upload(wide), device.upload(pick), device.upload(wts)
    out, head = device.zeros((R, D), torch.float32), device.zeros((short, D), torch.float32)
    pe.run(device.stream(), dx.data_ptr(), D + pad, dp.data_ptr(), dw.data_ptr(), ex, pe.Scratch(ex, R, 8, planes=planes),
           out.data_ptr(), R, do_round=False, x_dtype=x_dtype)
    pe.run(device.stream(), dx.data_ptr(), D + pad, dp.data_ptr(), dw.data_ptr(), ex,
           pe.Scratch(ex, short, 8, planes=planes), head.data_ptr(), short, do_round=False, x_dtype=x_dtype)
    got = device.download(out)
    assert_close_rms(got, orc.prompt_experts(x, pick, wts, oracle_routed(host), R, 8, bf16=x_dtype == 1), 2e-3, "long pass")
    np.testing.assert_array_equal(got[:short], device.download(head))
    assert device.device_status() == 0


@pytest.mark.parametrize("R,D,I,slots,k2", [(270, 256, 512, 8, 8), (520, 256, 512, 8, 6), (300, 512, 1024, 8, 10),
                                            (1100, 512, 256, 2, 8), (1030, 512, 384, 8, 5)])
def test_prompt_experts_gate_up_forms(ea, R, D, I, slots, k2):
    """The larger items' gate|up in two buffers, in one, and in one on four waves a SIMD (chosen by rows and by pairs times the
    intermediate's width), the down product of intermediates above 256, and more than 1,024 rows of few slots (rotated by
    a launch): the oracle's bar, and a row's bits are those of the same row in a short pass."""
    device, _, moe, pe, synth = ea
    E, short = 24, 60
    pick, wts = synth.picks_zipf(660 + R, R, 1.1, E, slots), synth.routing_weights(661, R, slots)
    host = synth.HostLayer(662, experts=E, dims=D, width=I, k2=k2, cb=1)
    x = synth.activations(663, R, D, "bf16")
    ex = moe.Routed(host)
    dx, dp, dw = device.upload(x), device.upload(pick), device.upload(wts)
    got = []
    for rows in (R, short):
        out = device.zeros((rows, D), torch.float32)
        pe.run(device.stream(), dx.data_ptr(), D, dp.data_ptr(), dw.data_ptr(), ex, pe.Scratch(ex, rows, slots), out.data_ptr(),
               rows, do_round=False)
        got.append(device.download(out))
    want = orc.prompt_experts(x, pick, wts, oracle_routed(host), R, slots, bf16=True)
    assert_close_rms(got[0], want, 2e-3, f"R={R} I={I} slots={slots}")
    np.testing.assert_array_equal(got[0][:short], got[1])
    assert device.device_status() == 0


def test_prompt_experts_second_chunk(ea):
    """More than 4,096 rows: the second chunk of rows takes the same scratch after the first. With and without the pair plane
    (whose down rows then lie where the second chunk's rotated inputs go) the same bits, and those of the second chunk's
    rows in a call of their own."""
    device, _, _, pe, synth = ea
    R, E, D, I, cut = 4300, 32, 256, 128, 4096
    host, ex, sc, x, pick, wts, dx, dp, dw = _prompt_case(ea, R, E, D, I, 8, 640, planes=False)
    got = []
    for s in (sc, pe.Scratch(ex, R, 8, planes=True)):
        out = device.zeros((R, D), torch.float32)
        pe.run(device.stream(), dx.data_ptr(), D, dp.data_ptr(), dw.data_ptr(), ex, s, out.data_ptr(), R, do_round=False)
        got.append(device.download(out))
    np.testing.assert_array_equal(got[0], got[1])
    tail = device.zeros((R - cut, D), torch.float32)
    pe.run(device.stream(), dx.data_ptr() + cut * D * 2, D, dp.data_ptr() + cut * 32, dw.data_ptr() + cut * 32, ex, sc,
           tail.data_ptr(), R - cut, do_round=False)
    np.testing.assert_array_equal(device.download(tail), got[0][cut:])
    rows = np.concatenate([np.arange(0, R, 16), [cut - 1, cut, R - 1]])
    want = orc.prompt_experts(np.ascontiguousarray(x[rows]), np.ascontiguousarray(pick[rows]), np.ascontiguousarray(wts[rows]),
                              oracle_routed(host), len(rows), 8, bf16=True)
    assert_close_rms(got[0][rows], want, 2e-3, "two chunks (sampled rows)")
    assert device.device_status() == 0


@pytest.mark.parametrize("planes", [True, False])
def test_prompt_experts_f32_activations(ea, planes):
    """fp32 activations (x_dtype 2: the rotation launch reads them and rounds the rotated rows to fp16 as for 16-bit
    ones), with the pair plane and without it, against the oracle on the same fp32 rows."""
    device, _, _, pe, synth = ea
    R, E, D, I = 96, 32, 512, 256
    host, ex, sc, x, pick, wts, dx, dp, dw = _prompt_case(ea, R, E, D, I, 8, 700 + int(planes), x_dtype=2,
                                                          planes=planes)
    assert x.dtype == np.float32
    want = orc.prompt_experts(x, pick, wts, oracle_routed(host), R, 8)
    out = device.zeros((R, D), torch.float32)
    pe.run(device.stream(), dx.data_ptr(), D, dp.data_ptr(), dw.data_ptr(), ex, sc, out.data_ptr(), R,
           do_round=False, x_dtype=2)
    assert_close_rms(device.download(out), want, 2e-3, f"prompt experts, fp32 x, planes={planes}")
    assert device.device_status() == 0


@pytest.mark.parametrize("cb,I", [(0, 256), (2, 256), (2, 128), (0, 128)])
def test_prompt_experts_codebooks(ea, cb, I):
    """3inst and mul1 through both item lists (the small items' ring kernel and the larger items' kernel), one and two
    column blocks of 128 in the intermediate."""
    device, _, _, pe, synth = ea
    R, E, D = 160, 48, 512
    host, ex, sc, x, pick, wts, dx, dp, dw = _prompt_case(ea, R, E, D, I, 8, 500 + cb + I, cb=cb)
    want = orc.prompt_experts(x, pick, wts, oracle_routed(host), R, 8, bf16=True)
    out = device.zeros((R, D), torch.float32)
    pe.run(device.stream(), dx.data_ptr(), D, dp.data_ptr(), dw.data_ptr(), ex, sc, out.data_ptr(), R, do_round=False)
    assert_close_rms(device.download(out), want, 2e-3, f"prompt experts cb={cb}")
    assert device.device_status() == 0


def test_prompt_unaligned_output_same_bits(ea):
    """An output 4 bytes off a 16-byte boundary is stored 4 bytes at a time: the same bits as 16 at a time."""
    device, _, _, pe, synth = ea
    R, D = 40, 512
    host, ex, sc, x, pick, wts, dx, dp, dw = _prompt_case(ea, R, 32, D, 128, 8, 400)
    a = device.zeros((R, D), torch.float32)
    pe.run(device.stream(), dx.data_ptr(), D, dp.data_ptr(), dw.data_ptr(), ex, sc, a.data_ptr(), R, do_round=False)
    b = device.zeros((R * D + 4,), torch.float32)
    pe.run(device.stream(), dx.data_ptr(), D, dp.data_ptr(), dw.data_ptr(), ex, sc, b.data_ptr() + 4, R,
           do_round=False)
    np.testing.assert_array_equal(device.download(b)[1:1 + R * D].reshape(R, D), device.download(a))
    assert device.device_status() == 0


def test_prompt_half_sums_and_invalid(ea):
    """half_sums is the reference's mode 1: no pair plane, an fp16 out (prompt_experts.zig:150-155, prompt_experts.cu:785-797,
    which adds each slot into it; here the fp32 sum of the slots is rounded once). Refused with rounding
    (prompt_experts.zig:147) and with a pair plane (:155). The bits are those of the fp32 output rounded to fp16."""
    device, _, _, pe, synth = ea
    from ea_exl3._lib import EaError

    R, D = 20, 256
    host, ex, sc, x, pick, wts, dx, dp, dw = _prompt_case(ea, R, 16, D, 128, 8, 300, planes=False)
    out = device.zeros((R, D), torch.float32)
    with pytest.raises(EaError) as e:  # prompt_experts.zig:147: half sums and rounding together
        pe.run(device.stream(), dx.data_ptr(), D, dp.data_ptr(), dw.data_ptr(), ex, sc, out.data_ptr(), R,
               do_round=True, half_sums=True)
    assert e.value.code == 13
    sc_plane = pe.Scratch(ex, R, 8, planes=True)
    with pytest.raises(EaError) as e:  # prompt_experts.zig:155: the pair plane takes fp32 rows only
        pe.run(device.stream(), dx.data_ptr(), D, dp.data_ptr(), dw.data_ptr(), ex, sc_plane, out.data_ptr(), R,
               do_round=False, half_sums=True)
    assert e.value.code == 13
    pick2 = pick.copy()
    pick2[0, 3] = -1  # a slot that is not an expert adds nothing
    want = orc.prompt_experts(x, pick2, wts, oracle_routed(host), R, 8, bf16=True)
    h = device.zeros((R, D), torch.float16)
    h.fill_(7.0)  # what out holds does not matter
    dp2 = device.upload(pick2)
    pe.run(device.stream(), dx.data_ptr(), D, dp2.data_ptr(), dw.data_ptr(), ex, sc, h.data_ptr(), R,
           do_round=False, half_sums=True)
    pe.run(device.stream(), dx.data_ptr(), D, dp2.data_ptr(), dw.data_ptr(), ex, sc, out.data_ptr(), R, do_round=False)
    full = device.download(out)
    assert_close_rms(full, want, 2e-3, "fp32 sums, no plane, a slot without an expert")
    np.testing.assert_array_equal(device.download(h).view(np.uint16), synth.f16_bits(full))
    assert device.device_status() == 0


@pytest.mark.parametrize("R,E,D,I,k2", [(130, 64, 512, 256, 8), (300, 256, 1024, 256, "mixed"), (40, 32, 256, 128, 6),
                                        (300, 32, 256, 128, 12), (260, 32, 512, 256, "wide-mixed")])
def test_prompt_experts_no_plane(ea, R, E, D, I, k2):
    """planes = 0, the reference's default mode 0: no pair plane, the pairs' down rows over their rotated inputs. Both item
    lists, widths up to 10 and above; out starts dirty; do_round rounds the sums through bf16. Every run meets the oracle's
    bar and gives the bits of planes 1 (the same products, the slots added in the same order)."""
    device, _, _, pe, synth = ea
    if k2 == "wide-mixed":
        k2v = np.array([(12, 8, 6, 16, 10, 11, 4, 14)[e % 8] for e in range(E)], np.int32)
    else:
        k2v = synth.mixed_widths(5, E) if k2 == "mixed" else k2
    host, ex, sc, x, pick, wts, dx, dp, dw = _prompt_case(ea, R, E, D, I, k2v, 700 + R, planes=False)
    assert sc.c.plane == 0
    want = orc.prompt_experts(x, pick, wts, oracle_routed(host), R, 8, bf16=True)
    sc_plane = pe.Scratch(ex, R, 8, planes=True)
    ref = device.zeros((R, D), torch.float32)
    pe.run(device.stream(), dx.data_ptr(), D, dp.data_ptr(), dw.data_ptr(), ex, sc_plane, ref.data_ptr(), R,
           do_round=False)
    for rep in range(2):
        out = device.zeros((R, D), torch.float32)
        out.fill_(float("nan") if rep else 3.0)
        pe.run(device.stream(), dx.data_ptr(), D, dp.data_ptr(), dw.data_ptr(), ex, sc, out.data_ptr(), R,
               do_round=False)
        got = device.download(out)
        assert_close_rms(got, want, 2e-3, f"prompt experts, no plane, run {rep}")
        np.testing.assert_array_equal(got, device.download(ref), err_msg=f"no plane against the plane, run {rep}")
    pe.run(device.stream(), dx.data_ptr(), D, dp.data_ptr(), dw.data_ptr(), ex, sc, out.data_ptr(), R, do_round=True)
    r = device.download(out)
    np.testing.assert_array_equal(r, synth.bf16_to_f32(synth.bf16_bits(r)))  # every value a bf16
    # within the fp32 bar plus bf16's half ulp (2^-9 relative) of each value
    w64 = want.astype(np.float64)
    bound = 2e-3 * np.sqrt(np.mean(w64 ** 2)) + np.abs(w64) * 2.0 ** -8
    assert np.all(np.abs(r.astype(np.float64) - w64) <= bound), "no plane, rounded through bf16"
    assert device.device_status() == 0
