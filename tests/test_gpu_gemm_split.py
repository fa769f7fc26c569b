"""GEMMs whose output tiles are shared by several workgroups along K (gemm_frag.hpp), and the tiles and epilogues around
them (each by the name of its kernel), at the sizes where they can go wrong: one slice per part and uneven parts, ragged rows and columns, row lengths of
the output that are no whole vectors, a launch repeated on the same tickets, two streams at once, graph replays."""
import pytest

pytestmark = pytest.mark.gpu


def _inputs(seed, M, K, N):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def q8(shape):
        return torch.clamp(torch.round(torch.randn(shape, generator=g, device="cuda") * 40), -128, 127).to(torch.int8)
    return q8((M, K)), q8((K, N)), torch.rand(M, generator=g, device="cuda") * 0.01 + 0.005, torch.rand(N, generator=g, device="cuda") * 3e-4 + 1e-4


def _expect(a, w, a_s, w_s):
    acc = a.double() @ w.double()                      # |sums| < 2^31: exact
    return ((acc.float() * a_s[:, None]) * w_s[None, :]).half()


# (M, K, N): the host's estimate splits K in most of these (few tiles, many slices)
@pytest.mark.parametrize("shape", [(200, 12288, 512), (33, 2048, 40), (100, 4096, 300), (129, 11520, 257), (398, 11520, 1856), (65, 1152, 129),
                                   (700, 6528, 200), (1000, 8064, 1000), (256, 8192, 8), (40, 14336, 2051)])
def test_w8a8_split_tiles_are_exact(pkg, shape):
    """Integer sums: bit-exact whatever the number of parts, and the same without scratch memory (unsplit)."""
    import torch
    M, K, N = shape
    a, w, a_s, w_s = _inputs(M + K + N, M, K, N)
    wf = pkg.gemm_w8a8_prepack_fragments(w)
    expect = _expect(a, w, a_s, w_s)
    for _ in range(3):                                 # the tickets are back at zero after each launch
        assert torch.equal(pkg.gemm_w8a8_fragments(a, wf, a_s, w_s, N), expect)
    y = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
    L = pkg.lib()
    stream = torch.cuda.current_stream().cuda_stream
    pkg.check(L.mtrt_hip_gemm_w8a8_fragments(stream, a.data_ptr(), wf.data_ptr(), a_s.data_ptr(), w_s.data_ptr(), y.data_ptr(), M, K, N))
    assert torch.equal(y, expect)
    need = L.mtrt_hip_gemm_w8a8_fragments_workspace(M, K, N)
    if need:                                           # one byte too few: the unsplit form again
        scratch = torch.empty(need, dtype=torch.uint8, device="cuda")
        y.fill_(float("nan"))
        pkg.check(L.mtrt_hip_gemm_w8a8_fragments_ws(stream, a.data_ptr(), wf.data_ptr(), a_s.data_ptr(), w_s.data_ptr(), y.data_ptr(), M, K, N,
                                                    scratch.data_ptr(), need - 1))
        assert torch.equal(y, expect)


def test_some_shape_is_split(pkg):
    L = pkg.lib()
    assert L.mtrt_hip_gemm_w8a8_fragments_workspace(200, 12288, 512) > 0
    assert L.mtrt_hip_gemm_w8a8_fragments_workspace(16, 12288, 512) == 0 and L.mtrt_hip_gemm_w8a8_fragments_workspace(200, 128, 512) == 0


@pytest.mark.parametrize("N", [8, 12, 129, 1001, 2048 + 6])
@pytest.mark.parametrize("M", [65, 300, 1100, 2100])
def test_w8a8_outputs_inside_a_larger_buffer(pkg, M, N):
    """Row lengths that are no whole 16-byte vectors and outputs off 16-byte alignment: the results are exact and nothing
    around them is written."""
    import torch
    K = 256
    a, w, a_s, w_s = _inputs(M * N, M, K, N)
    wf = pkg.gemm_w8a8_prepack_fragments(w)
    buf = torch.full((M * N + 9,), 7.0, dtype=torch.float16, device="cuda")
    y = buf[1:1 + M * N].view(M, N)
    pkg.gemm_w8a8_fragments(a, wf, a_s, w_s, N, out=y)
    assert torch.equal(y, _expect(a, w, a_s, w_s))
    assert float(buf[0]) == 7.0 and bool((buf[1 + M * N:] == 7.0).all())


def test_w8a8_split_launches_on_two_streams_and_in_a_graph(pkg):
    """Tickets belong to a stream: launches on two streams do not meet; a captured launch gives the eager result on every
    replay, with eager work between the replays."""
    import torch
    cases = [_inputs(k, 200, 12288, 512) for k in range(2)]
    frag = [pkg.gemm_w8a8_prepack_fragments(w) for _, w, _, _ in cases]
    expect = [_expect(*c) for c in cases]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    out = [[], []]
    for _ in range(8):
        for k, s in enumerate(streams):
            with torch.cuda.stream(s):
                a, _, a_s, w_s = cases[k]
                out[k].append(pkg.gemm_w8a8_fragments(a, frag[k], a_s, w_s, 512))
    torch.cuda.synchronize()
    assert all(torch.equal(y, expect[k]) for k in range(2) for y in out[k])
    a, _, a_s, w_s = cases[0]
    static = a.clone()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        pkg.gemm_w8a8_fragments(static, frag[0], a_s, w_s, 512)      # the stream's block is bound before the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        y = pkg.gemm_w8a8_fragments(static, frag[0], a_s, w_s, 512)
    for k in range(4):
        static.copy_(torch.roll(a, k, 0))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, pkg.gemm_w8a8_fragments(static, frag[0], a_s, w_s, 512)), k


def test_graphs_recorded_on_one_stream_replay_at_once(pkg):
    """Two graphs recorded on the same stream, replayed together on two others, with eager launches on the recording stream beside
    them: every launch has tickets of its own, so each result is the eager one."""
    import importlib

    import torch
    tp = importlib.import_module(pkg.__name__ + ".tp")
    a8, w8, a_s, w_s = _inputs(5, 200, 12288, 512)
    f8 = pkg.gemm_w8a8_prepack_fragments(w8)
    a4, packed, s4, _ = _w4_inputs(6, 64, 8256, 96, 64)
    p4 = pkg.gemm_w4a16_prepack(packed, 8256, 96)
    lin = tp.Linear(11520, 320, dtype=tp.float16)
    lin.weight = tp.Tensor((torch.randn(320, 11520) * 0.05).half())
    x = torch.randn(100, 11520).half().cuda()

    def calls(shift):
        return [pkg.gemm_w8a8_fragments(a8.roll(shift, 0), f8, a_s, w_s, 512),
                pkg.gemm_w4a16(a4.roll(shift, 0), s4, 8256, 96, 64, w_prepacked=p4), lin(tp.Tensor(x.roll(shift, 0))).torch()]
    want = [calls(k) for k in range(3)]
    torch.cuda.synchronize()
    record, streams = torch.cuda.Stream(), [torch.cuda.Stream(), torch.cuda.Stream()]
    graphs, results = [torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()], [[], []]
    for k in range(2):
        with torch.cuda.graph(graphs[k], stream=record):             # a memory pool each
            for _ in range(10):
                results[k] += calls(k)
    for replay in range(4):
        for y in results[0] + results[1]:
            y.zero_()
        torch.cuda.synchronize()
        for k in range(2):
            with torch.cuda.stream(streams[k]):
                graphs[k].replay()
        with torch.cuda.stream(record):
            eager = [y for _ in range(5) for y in calls(2)]
        torch.cuda.synchronize()
        for ys, expect, who in ((results[0], want[0], "first graph"), (results[1], want[1], "second graph"), (eager, want[2], "eager")):
            for i, y in enumerate(ys):
                assert torch.equal(y, expect[i % 3]), (replay, who, i)


def _w4_inputs(seed, M, K, N, B):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    a = torch.randn((M, K), generator=g, device="cuda").half()
    q = torch.randint(-8, 8, (K, N), generator=g, device="cuda")
    s = (torch.rand((K // B, N), generator=g, device="cuda") * 0.02 + 0.005).half()
    nibbles = (q & 15).to(torch.uint8).reshape(-1)
    if nibbles.numel() % 2:
        nibbles = torch.cat([nibbles, nibbles.new_zeros(1)])
    return a, (nibbles[0::2] | (nibbles[1::2] << 4)).contiguous(), s, (q.half() * s.repeat_interleave(B, 0)).double()


# (M, K, N, block): split and not, ragged rows and columns, blocks of one slice and of all of K
@pytest.mark.parametrize("case", [(33, 4096, 200, 128), (48, 2048, 1000, 64), (64, 8192, 96, 8192), (65, 1152, 129, 192), (100, 12288, 300, 128),
                                  (130, 4096, 4096, 128), (200, 384, 8, 64), (256, 8192, 2051, 256), (300, 4096, 3000, 128), (600, 256, 40, 64),
                                  (700, 4864, 60, 128), (1000, 640, 2000, 128), (1800, 640, 1160, 128), (517, 64, 472, 64), (2000, 2048, 769, 128)])
def test_w4a16_tiles_and_splits(pkg, case):
    """Against float64 on the dequantised weights: products exact, f32 sums in any order, one rounding to f16; nothing
    around the output is written; the same bits on every launch."""
    import torch
    M, K, N, B = case
    a, packed, s, wd = _w4_inputs(M + K + N, M, K, N, B)
    pre = pkg.gemm_w4a16_prepack(packed, K, N)
    ref, mass = a.double() @ wd, a.double().abs() @ wd.abs()
    tol = 2.0 ** -11 * ref.abs() + (1 + 2.0 ** -11) * (K + 1) * 2.0 ** -24 * mass + 2.0 ** -25

    buf = torch.full((M * N + 9,), 7.0, dtype=torch.float16, device="cuda")
    y = buf[1:1 + M * N].view(M, N)
    pkg.gemm_w4a16(a, s, K, N, B, w_prepacked=pre, out=y)
    assert bool(((y.double() - ref).abs() <= tol).all()) and float(buf[0]) == 7.0 and bool((buf[1 + M * N:] == 7.0).all())
    for _ in range(3):
        assert torch.equal(pkg.gemm_w4a16(a, s, K, N, B, w_prepacked=pre), y)
    L = pkg.lib()
    need = L.mtrt_hip_gemm_w4a16_workspace(M, K, N, B)
    z = torch.empty((M, N), dtype=torch.float16, device="cuda")
    scratch = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    pkg.check(L.mtrt_hip_gemm_w4a16_ws(stream, a.data_ptr(), None, pre.data_ptr(), s.data_ptr(), z.data_ptr(), M, K, N, B, scratch.data_ptr(),
                                       need - 1 if need else 0))                     # too little: unsplit
    assert bool(((z.double() - ref).abs() <= tol).all())


def test_some_w4a16_shape_is_split(pkg):
    L = pkg.lib()
    assert L.mtrt_hip_gemm_w4a16_workspace(64, 8256, 96, 64) > 0
    assert L.mtrt_hip_gemm_w4a16_workspace(32, 8192, 96, 128) == 0 and L.mtrt_hip_gemm_w4a16_workspace(64, 8192, 96, 96) == 0


# A shape with ragged rows and columns for each tile, with its K whole and shared, as the host's estimate picks them on 256 compute
# units; `workspace` says whether K is shared.  The tiles wider or higher than 128 x 256 with an odd number of slices too.
W8_TILES = [((41, 256, 9), "t32x128", 0), ((41, 3584, 9), "t32x128", 1), ((2115, 256, 387), "t64x128", 0), ((2849, 11904, 9), "t64x128", 1),
            ((2143, 256, 913), "t128x128", 0), ((1187, 8704, 793), "t128x128", 1), ((323, 256, 10933), "t128x256", 0),
            ((1647, 8448, 1253), "t128x256", 1), ((2563, 768, 3171), "t128x384", 0), ((2747, 12160, 1423), "t128x384", 1),
            ((2545, 2304, 4683), "t256x256", 0), ((1669, 512, 9249), "t256x384", 0), ((661, 896, 10901), "t128x384", 0),
            ((2488, 2944, 4629), "t256x256", 0), ((1296, 640, 12203), "t256x384", 0)]
W4_TILES = [((45, 704, 9), "t32x128", 0), ((41, 1344, 9), "t32x128", 1), ((133, 640, 10297), "t64x128", 0), ((2791, 4736, 9), "t64x128", 1),
            ((261, 256, 9955), "t64x256", 0), ((1027, 6592, 963), "t64x256", 1), ((8389, 64, 13), "t128x64", 0), ((1387, 64, 1287), "t128x128", 0),
            ((2727, 5248, 279), "t128x128", 1), ((385, 64, 8453), "t128x256", 0), ((665, 256, 11017), "t256x256", 0), ((1497, 256, 10781), "t256x384", 0)]
DENSE_TILES = [((41, 64, 9), "t32x128", 0), ((53, 1792, 9), "t32x128", 1), ((2115, 256, 387), "t64x128", 0), ((2781, 5568, 9), "t64x128", 1),
               ((2143, 256, 913), "t128x128", 0), ((2727, 5248, 279), "t128x128", 1), ((323, 256, 10933), "t128x256", 0),
               ((2701, 4544, 657), "t128x256", 1), ((2399, 384, 3391), "t128x384", 0), ((143, 9024, 11467), "t128x384", 1),
               ((2473, 1152, 4611), "t256x256", 0), ((1497, 256, 10781), "t256x384", 0), ((1055, 576, 7361), "t128x384", 0),
               ((5433, 1472, 2039), "t256x256", 0), ((2787, 64, 8713), "t256x384", 0), ((1671, 320, 9275), "t256x384", 0)]


def _is(pkg, kernel):
    import torch
    assert torch.cuda.get_device_properties(0).multi_processor_count != 256 or pkg.last_kernel() == kernel, pkg.last_kernel()


@pytest.mark.parametrize("shape,tile,split", W8_TILES)
def test_every_w8a8_tile(pkg, shape, tile, split):
    import torch
    M, K, N = shape
    a, w, a_s, w_s = _inputs(M + N, M, K, N)
    wf = pkg.gemm_w8a8_prepack_fragments(w)
    y = pkg.gemm_w8a8_fragments(a, wf, a_s, w_s, N)
    _is(pkg, "mtrt_gemm_w8a8_frag_" + tile)
    assert (pkg.lib().mtrt_hip_gemm_w8a8_fragments_workspace(M, K, N) > 0) == bool(split)
    assert torch.equal(y, _expect(a, w, a_s, w_s))


@pytest.mark.parametrize("shape,tile,split", W4_TILES)
def test_every_w4a16_tile(pkg, shape, tile, split):
    """The bound of test_w4a16_tiles_and_splits; with a bias (a Linear with one scale per output) one more rounding."""
    import importlib

    import torch
    tp = importlib.import_module(pkg.__name__ + ".tp")
    M, K, N = shape
    a, packed, s, wd = _w4_inputs(M + N, M, K, N, 64)
    y = pkg.gemm_w4a16(a, s, K, N, 64, w_prepacked=pkg.gemm_w4a16_prepack(packed, K, N))
    _is(pkg, "mtrt_gemm_w4a16_" + tile)
    assert (pkg.lib().mtrt_hip_gemm_w4a16_workspace(M, K, N, 64) > 0) == bool(split)
    ref, mass = a.double() @ wd, a.double().abs() @ wd.abs()
    tol = 2.0 ** -11 * ref.abs() + (1 + 2.0 ** -11) * (K + 1) * 2.0 ** -24 * mass + 2.0 ** -25
    assert bool(((y.double() - ref).abs() <= tol).all())

    lin = tp.Linear(K, N, dtype=tp.float16, quant_dtype=tp.int4, weight_quant_dim=0)
    q = torch.randint(-8, 8, (N, K)).half()
    s_w, b = torch.rand(N).half() * 0.02 + 0.005, torch.randn(N).half()
    lin.load_state_dict({"weight": tp.Tensor(q * s_w[:, None]), "weight_scale": tp.Tensor(s_w), "bias": tp.Tensor(b)})
    y = lin(tp.Tensor(a)).torch()
    assert lin.route() == "w4a16"
    _is(pkg, "mtrt_gemm_w4a16_%s_bias" % tile)
    wd = (tp.quantize(lin.weight, lin.weight_scale, tp.int4, 0).torch().to(torch.int8) << 4 >> 4).half() * s_w.cuda()[:, None]
    core, mass = a.double() @ wd.double().T, a.double().abs() @ wd.double().abs().T
    ref, u = core + b.cuda().double(), 2.0 ** -11
    tol = u * core.abs() + (1 + u) * (K + 2) * 2.0 ** -24 * mass + u * ref.abs() * (1 + u) + 2.0 ** -24
    assert bool(((y.double() - ref).abs() <= tol).all())


# Sets of waves that take slices in turn: parts with a whole number of rounds and each rest, the last part of a split another one
# than the others, ragged rows and columns; blocks of one, two, three and four slices and one block for all.
@pytest.mark.parametrize("shape,tile,blocks", [
    ((513, 1152, 130), "t32x128x2", (64, 128, 192, 1152)), ((40, 1088, 130), "t32x128x2", (64,)), ((63, 8768, 130), "t32x128x2", (64,)), ((65, 8256, 130), "t32x128x2", (64, 192)),
    ((33, 2304, 8641), "t32x128x4", (64, 128, 192, 256, 2304)), ((33, 2368, 8641), "t32x128x4", (64,)), ((33, 2176, 8641), "t32x128x4", (128,)),
    ((97, 2240, 4100), "t32x128x4", (64, 320)), ((33, 9024, 3000), "t32x128x4", (64, 192)), ((33, 6848, 4100), "t32x128x4", (64,)),
    ((130, 1152, 8000), "t64x128", (64, 128, 192, 1152)), ((97, 1216, 8641), "t64x128", (64,)), ((33, 2688, 8641), "t64x128", (64, 128)), ((40, 2496, 8641), "t64x128", (192,))])
def test_w4a16_slices_in_turn(pkg, shape, tile, blocks):
    import torch
    M, K, N = shape
    for block in blocks:
        a, packed, s, wd = _w4_inputs(M + block, M, K, N, block)
        a[3, 0], a[4, K - 1] = float("inf"), float("-inf")     # a slice counts once: no infinity of another's, none that cancels
        y = pkg.gemm_w4a16(a, s, K, N, block, w_prepacked=pkg.gemm_w4a16_prepack(packed, K, N)).double()
        _is(pkg, "mtrt_gemm_w4a16_" + tile)
        for row, k, sign in ((3, 0, 1.0), (4, K - 1, -1.0)):
            assert torch.equal(y[row].nan_to_num(7.0, posinf=1.0, neginf=-1.0), torch.where(wd[k] == 0, torch.full_like(wd[k], 7.0), sign * wd[k].sign()))
        a[3:5], y[3:5] = 0, 0
        ref, mass = a.double() @ wd, a.double().abs() @ wd.abs()
        assert bool(((y - ref).abs() <= 2.0 ** -11 * ref.abs() + (1 + 2.0 ** -11) * (K + 1) * 2.0 ** -24 * mass + 2.0 ** -25).all()), block


@pytest.mark.parametrize("dname", ["float16", "bfloat16"])
@pytest.mark.parametrize("shape,tile,split", DENSE_TILES)
def test_every_dense_tile(pkg, shape, tile, split, dname):
    import importlib

    import torch
    tp = importlib.import_module(pkg.__name__ + ".tp")
    M, K, N = shape
    td, u = getattr(torch, dname), {"float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}[dname]
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N)
    x, w, b = (torch.randn(s, generator=g, device="cuda").to(td) for s in ((M, K), (N, K), (N,)))
    lin = tp.Linear(K, N, dtype=getattr(tp, dname))
    lin.weight, lin.bias = tp.Tensor(w), tp.Tensor(b)
    y = lin(tp.Tensor(x)).torch()
    _is(pkg, "mtrt_gemm_dense_frag_%s_%s" % ({"float16": "f16", "bfloat16": "bf16"}[dname], tile))
    ref, mass = x.double() @ w.double().T + b.double(), x.double().abs() @ w.double().abs().T + b.double().abs()
    assert bool(((y.double() - ref).abs() <= u * ref.abs() + (1 + u) * (K + 2) * 2.0 ** -24 * mass + 2.0 ** -24).all())


# More than one 128 x 256 tile to a compute unit, which two workgroups share; rows that are whole cache lines, whole vectors and neither.
@pytest.mark.parametrize("N", [5376, 5384, 5391])
def test_pairs_of_tiles_on_a_unit(pkg, N):
    import importlib

    import torch
    tp = importlib.import_module(pkg.__name__ + ".tp")
    M = 2817
    a, w, a_s, w_s = _inputs(N, M, 768, N)
    y = pkg.gemm_w8a8_fragments(a, pkg.gemm_w8a8_prepack_fragments(w), a_s, w_s, N)
    _is(pkg, "mtrt_gemm_w8a8_frag_t128x256")
    assert torch.equal(y, _expect(a, w, a_s, w_s))
    x, w, b = (torch.randn(s, device="cuda").half() for s in ((M, 384), (N, 384), (N,)))
    lin = tp.Linear(384, N, dtype=tp.float16)
    lin.weight, lin.bias = tp.Tensor(w), tp.Tensor(b)
    y = lin(tp.Tensor(x)).torch()
    _is(pkg, "mtrt_gemm_dense_frag_f16_t128x256")
    ref, mass, u = x.double() @ w.double().T + b.double(), x.double().abs() @ w.double().abs().T + b.double().abs(), 2.0 ** -11
    assert bool(((y.double() - ref).abs() <= u * ref.abs() + (1 + u) * (384 + 2) * 2.0 ** -24 * mass + 2.0 ** -24).all())
