"""The 32x32-tile GEMM (more than 16 activation rows) in each of its tile
shapes, at the edges of tiles, segments and shares of K.

Oracle: the exact int32 I of the oracle, scaled and summed in float64. An
output is one rounding per sub-block product, at most four per 128-column
block inside it, one per block of a share's chain and one per share, so
    |y - y64| <= (nblocks + 16) * 2^-24 * sum |scale * d * I|
(each rounding is at most 2^-24 of a partial sum that the sum of magnitudes
bounds); swiglu adds its own few roundings (2^-20 of the product's bound,
expf within 2 ulp, and the derivative of silu below 1.1).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _torch():
    import torch
    return torch


def dev(a):
    torch = _torch()
    a = np.ascontiguousarray(a)
    if a.dtype == np.uint16:
        a = a.view(np.int16)
    return torch.from_numpy(a.copy()).cuda()


def stream():
    return _torch().cuda.current_stream().cuda_stream


def matrix(rng, N, K):
    """Codes with P(-1, 0, +1) = (0.3, 0.4, 0.3) and scales in [0.01, 0.05]."""
    c = rng.choice(3, p=[0.3, 0.4, 0.3], size=(4096, 4)).astype(np.uint8)
    lut = c[:, 0] | c[:, 1] << 2 | c[:, 2] << 4 | c[:, 3] << 6
    codes = lut[rng.integers(0, 4096, (N, K // 4))]
    scales = (0.01 + 0.04 * rng.random((N, K // 128))).astype(np.float16).view(np.uint16)
    return codes, scales


def wide(oracle, mat, sel, K, q, d, s):
    """(y, sum of magnitudes) of the sampled rows in float64, [M][len(sel)]."""
    codes, scales = np.ascontiguousarray(mat[0][sel]), mat[1][sel].view(np.float16).astype(np.float64)
    I = oracle.gemv_i32(codes, K, q, s).astype(np.float64)
    t = I * d.astype(np.float64)[:, None, :] * np.repeat(scales, 4, axis=1)[None]
    return t.sum(-1), np.abs(t).sum(-1)


# (K, M, Ns, swiglu N): tiles of 32 x 32 outputs, by which the launch chooses. K has four
# shares below 4096, eight from there.
CASES = [
    (128, 17, [1, 33], 1),           # one activation tile with 15 dead rows, one block: three of four K groups have none
    (256, 32, [16070, 5], 8030),     # 504 / 502 tiles of few blocks: one wave x four groups, one full activation tile
    (128, 25, [131105], 65600),      # 4098 / 4100 tiles of one activation tile: four waves, K unsplit
    (384, 64, [37, 70, 9], 17),      # three blocks over four groups, three segments
    (1152, 95, [45], 50),            # one wave x four groups, nine blocks: uneven groups, a dead row in the last tile
    (1152, 32, [8161], 4081),        # 256 / 256 tiles: the last of one tile per workgroup
    (1152, 32, [8193], 4097),        # 257 / 257 tiles: two waves x four groups
    (12416, 40, [37, 5], 20),        # one wave x eight groups, 97 blocks
    (4224, 64, [4200], 2200),        # 264 / 276 tiles: two waves x eight groups, 33 blocks
    (640, 65, [6917], 3500),         # 651 / 657 tiles: two waves x four groups; five blocks
    (640, 32, [16070, 5], 8030),     # the same of one full activation tile
    (4224, 40, [16100, 20], 8100),   # 1008 / 1014 tiles: two waves x four groups of two shares
    (2176, 40, [9000], 4500),        # 564 / 564 tiles: two waves x four groups of one share, 17 blocks
    (512, 520, [2000], 1000),        # 1071 / 1071 tiles of few blocks: four waves, K unsplit
    (1152, 1000, [3000], 1500),      # 3008 / 3008 tiles: four waves, K unsplit, four shares
    (4224, 900, [3000], 1500),       # 2726 / 2726 tiles: the same, eight shares of four or five blocks
    (256, 200, [18733], 9400),       # 4102 / 4116 tiles: four waves, K unsplit
    (256, 513, [15500], 7800),       # 8245 / 8296 tiles: 64 activation rows a wave, the last tile nearly empty
    (4224, 513, [15500], 7800),      # the same, eight shares
]


@pytest.mark.parametrize("K,M,Ns,N2", CASES)
def test_t32_modes_and_edges(hip, oracle, K, M, Ns, N2):
    torch = _torch()
    G = hip.GemvMode
    rng = np.random.default_rng(K + M)
    x = (rng.standard_normal((M, K)) * np.exp(rng.standard_normal((M, 1)))).astype(np.float32)
    q, d, s = oracle.quantize_rows(x)
    act = hip.Q8Act(dev(q), dev(d), dev(s))
    nblk = K // 128

    def check(got, want, mag, what):
        bound = (nblk + 16) * 2.0 ** -24 * mag
        bad = np.argwhere(np.abs(got.astype(np.float64) - want) > bound)
        assert bad.size == 0, f"{what}: {len(bad)} outputs past the bound, first {bad[0]}"

    def sample(N):
        return np.unique(np.r_[0:min(N, 40), max(0, N // 2 - 20):N // 2, max(0, N - 40):N])

    mats = [matrix(rng, n, K) for n in Ns]
    ys = [torch.full((M, n + 3), 7.0, device="cuda") for n in Ns]
    segs = [hip.GemvSeg(dev(c), dev(sc), n, y, n + 3) for (c, sc), n, y in zip(mats, Ns, ys)]
    hip.launch_gemv(segs, K, M, act, G.kStore, stream())
    for mat, n, y in zip(mats, Ns, ys):
        sel = sample(n)
        want, mag = wide(oracle, mat, sel, K, q, d, s)
        got = y.cpu().numpy()
        check(got[:, sel], want, mag, f"store N={n}")
        assert np.all(got[:, n:] == 7.0), "wrote past N"

    y0 = rng.standard_normal((M, Ns[0])).astype(np.float32)
    y = dev(y0)
    hip.launch_gemv([hip.GemvSeg(segs[0].codes, segs[0].scales, Ns[0], y, Ns[0])], K, M, act, G.kAdd, stream())
    sel = sample(Ns[0])
    want, mag = wide(oracle, mats[0], sel, K, q, d, s)
    check(y.cpu().numpy()[:, sel], want + y0[:, sel], mag + np.abs(y0[:, sel]), "add")

    gate, up = matrix(rng, N2, K), matrix(rng, N2, K)
    y = torch.full((M, N2 + 1), 7.0, device="cuda")
    hip.launch_gemv([hip.GemvSeg(dev(gate[0]), dev(gate[1]), N2, y, N2 + 1),
                     hip.GemvSeg(dev(up[0]), dev(up[1]), N2, None, 0)], K, M, act, G.kSwiglu, stream())
    sel = sample(N2)
    g, gm = wide(oracle, gate, sel, K, q, d, s)
    u, um = wide(oracle, up, sel, K, q, d, s)
    silu = g / (1 + np.exp(-g))
    got = y.cpu().numpy()
    bound = (nblk + 16) * 2.0 ** -24 * (1.1 * gm * np.abs(u) + np.abs(silu) * um) * 1.01 + 2.0 ** -20 * np.abs(silu * u)
    bad = np.argwhere(np.abs(got[:, sel] - silu * u) > bound)
    assert bad.size == 0, f"swiglu: {len(bad)} outputs past the bound, first {bad[0]}"
    assert np.all(got[:, N2:] == 7.0), "wrote past N"

    n = min(Ns[-1], 70)  # I of the exact dump, the tile chosen as for a launch of that size
    I = torch.full((M, n, K // 32), -(1 << 30), dtype=torch.int32, device="cuda")
    hip.gemv_i32_dump(dev(mats[-1][0][:n]), n, K, M, act, I, stream())
    assert np.array_equal(I.cpu().numpy(), oracle.gemv_i32(np.ascontiguousarray(mats[-1][0][:n]), K, q, s))


# one launch for each tile: (tile, K, M, N)
DUMPS = [((1, 1, 4), 128, 17, 45), ((1, 1, 8), 4224, 40, 45), ((1, 2, 8), 4224, 64, 4200), ((1, 2, 4), 640, 40, 8205),
         ((1, 4, 1), 128, 513, 2005), ((2, 4, 1), 128, 513, 15500)]


@pytest.mark.parametrize("tile,K,M,N", DUMPS)
def test_t32_exact_dump_in_each_tile(hip, oracle, tile, K, M, N):
    """The exact I, written by the tile that a launch of that size takes."""
    torch = _torch()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert cus != 256 or hip.gemm_tile(cus, [N], K, M) == tile
    rng = np.random.default_rng(K + M + N)
    q, d, s = oracle.quantize_rows((rng.standard_normal((M, K)) * 2).astype(np.float32))
    codes, _ = matrix(rng, N, K)
    I = torch.full((M, N, K // 32), -(1 << 30), dtype=torch.int32, device="cuda")
    hip.gemv_i32_dump(dev(codes), N, K, M, hip.Q8Act(dev(q), dev(d), dev(s)), I, stream())
    assert int(I.min()) > -(1 << 30), "outputs not written"
    sel = np.unique(np.r_[0:40, N // 2 - 20:N // 2 + 20, N - 40:N])
    got = I[:, torch.from_numpy(sel).cuda()].cpu().numpy()
    assert np.array_equal(got, oracle.gemv_i32(np.ascontiguousarray(codes[sel]), K, q, s))


@pytest.mark.parametrize("K,M,N", [(128, 17, 64), (1152, 24, 96), (12416, 20, 64), (4224, 20, 8480),
                                   (1152, 32, 8224), (256, 32, 16064), (128, 30, 131136),
                                   (128, 18, 262176), (256, 20, 32800)])
def test_t32_q8_output(hip, oracle, K, M, N):
    """launch_gemv_ex with a Q8 output in each tile shape of one activation
    tile: y equals launch_gemv's bit for bit, the Q8 rows equal the oracle's
    quantize of that y; the first block is all zero. y starts from values of
    its own, so that the add counts."""
    torch = _torch()
    rng = np.random.default_rng(K + M + N)
    q, d, s = oracle.quantize_rows((rng.standard_normal((M, K)) * 2).astype(np.float32))
    act = hip.Q8Act(dev(q), dev(d), dev(s))
    mats = [matrix(rng, N, K) for _ in range(2)]
    mats[0][0][:32] = 0x55  # trit 0
    w = [(dev(c), dev(sc)) for c, sc in mats]
    y0 = (rng.standard_normal((M, N)) * 8).astype(np.float32)
    y0[:, :32] = 0
    stored = None
    for mode in (hip.GemvMode.kStore, hip.GemvMode.kAdd, hip.GemvMode.kSwiglu):
        ys = []
        out = hip.Q8Act(torch.zeros((M, N), dtype=torch.int8, device="cuda"), torch.zeros((M, N // 32), device="cuda"),
                        torch.zeros((M, N // 32), dtype=torch.int32, device="cuda"))
        for fused in (False, True):
            y = dev(y0)
            segs = [hip.GemvSeg(*w[0], N, y, N)] + ([hip.GemvSeg(*w[1], N, None, 0)] if mode == 2 else [])
            if fused:
                hip.launch_gemv_ex(segs, K, M, act, mode=mode, out=out, stream=stream())
            else:
                hip.launch_gemv(segs, K, M, act, mode, stream())
            ys.append(y.cpu().numpy())
        assert np.array_equal(ys[0].view(np.uint32), ys[1].view(np.uint32)), f"y, mode {mode}"
        if mode == hip.GemvMode.kStore:
            stored = ys[1]
        elif mode == hip.GemvMode.kAdd:  # (more than 16 rows: the same sums as the store's)
            assert np.array_equal(ys[1], y0 + stored), "the old y is not in the sum"
        rq, rd, rs = oracle.quantize_rows(ys[1])
        assert np.array_equal(out.q.cpu().numpy(), rq), f"q, mode {mode}"
        assert np.array_equal(out.d.cpu().numpy().view(np.uint32), rd.view(np.uint32)), f"d, mode {mode}"
        assert np.array_equal(out.s.cpu().numpy(), rs), f"s, mode {mode}"


@pytest.mark.parametrize("K,N", [(1024, 2053), (1024, 1030), (5120, 33), (16384, 40), (16512, 2055), (16512, 4100),
                                 (17408, 20), (20480, 35), (20608, 18)])
def test_dot4_two_rows_equal_one_row_launches(hip, oracle, K, N):
    """Two activation rows on the v_dot4 path in one pass (both step counts,
    one and two chunks per lane, the widest rows one pass takes and the next
    wider) equal one-row launches bit for bit, and I equals the oracle's."""
    torch = _torch()
    rng = np.random.default_rng(K + N)
    q, d, s = oracle.quantize_rows((rng.standard_normal((2, K)) * 2).astype(np.float32))
    mats = [matrix(rng, N, K) for _ in range(2)]
    w = [(dev(c), dev(sc)) for c, sc in mats]
    y0 = rng.standard_normal((2, N)).astype(np.float32)
    for mode in (hip.GemvMode.kStore, hip.GemvMode.kAdd, hip.GemvMode.kSwiglu):
        def run(rows):
            y = dev(y0[rows])
            segs = [hip.GemvSeg(*w[0], N, y, N)] + ([hip.GemvSeg(*w[1], N, None, 0)] if mode == 2 else [])
            hip.launch_gemv(segs, K, len(rows), hip.Q8Act(dev(q[rows]), dev(d[rows]), dev(s[rows])), mode, stream())
            return y.cpu().numpy()
        both, single = run([0, 1]), np.concatenate([run([0]), run([1])])
        assert np.array_equal(both.view(np.uint32), single.view(np.uint32)), f"mode {mode}"
    I = torch.zeros((2, N, K // 32), dtype=torch.int32, device="cuda")
    hip.gemv_i32_dump(w[0][0], N, K, 2, hip.Q8Act(dev(q), dev(d), dev(s)), I, stream())
    assert np.array_equal(I.cpu().numpy(), oracle.gemv_i32(mats[0][0], K, q, s))


@pytest.mark.parametrize("K,wide_n", [(128, 9000), (640, 9000), (1152, 9000), (4224, 16390), (4992, 9000),
                                      (12416, 9000)])
def test_t32_rows_do_not_depend_on_the_launch(hip, K, wide_n):
    """More than 16 rows: an output's bits are the same however many rows and
    segments its launch has and in every tile shape that these choose, with
    gate and up in a swiglu too. K of one block, and of block counts that its
    shares do not divide; segments of four and of eight shares in one launch."""
    torch = _torch()
    G = hip.GemvMode
    rng = np.random.default_rng(K)
    M, N = 1000, 1030
    q = rng.integers(-127, 128, (M, K), dtype=np.int8)
    d = (0.001 + rng.random((M, K // 32)) * 0.05).astype(np.float16).astype(np.float32)
    s = q.reshape(M, K // 32, 32).sum(-1, dtype=np.int32)
    a, b, c = ([dev(t) for t in matrix(rng, n, K)] for n in (N, wide_n, N))

    def run(rows, mode, *mats):
        act = hip.Q8Act(dev(q[rows]), dev(d[rows]), dev(s[rows]))
        m = len(rows)
        ys = [torch.zeros((m, w[0].shape[0]), device="cuda") for w in mats]
        segs = [hip.GemvSeg(*w, w[0].shape[0], y, w[0].shape[0]) for w, y in zip(mats, ys)]
        hip.launch_gemv(segs, K, m, act, mode, stream())
        return [y.cpu().numpy().view(np.uint32) for y in ys]

    every = np.arange(M)
    ya, yb, yc = run(every, G.kStore, a, b, c)
    sw = run(every, G.kSwiglu, a, c)[0]
    for i, (y, w) in enumerate(((ya, a), (yb, b), (yc, c))):
        assert np.array_equal(run(every, G.kStore, w)[0], y), f"matrix {i} alone"
    # tiles of 32 x 32 outputs: 33 (a) and 315 (a and b of 9000) times a row group of 32
    for n in (17, 32, 40, 95, 200, 400, 513):
        rows = every[300:300 + n]
        assert np.array_equal(run(rows, G.kStore, a)[0], ya[rows]), f"{n} rows, one segment"
        got = run(rows, G.kStore, b, a)
        assert np.array_equal(got[0], yb[rows]) and np.array_equal(got[1], ya[rows]), f"{n} rows, two segments"
        assert np.array_equal(run(rows, G.kSwiglu, a, c)[0], sw[rows]), f"{n} rows, swiglu"
        assert np.array_equal(run(rows, G.kAdd, a)[0], ya[rows]), f"{n} rows, added to zeros"
