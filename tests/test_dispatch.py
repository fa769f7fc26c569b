"""What the entry points launch, seen on the CPU (dispatch.py): the words in which workgroups meet (tickets of K-split GEMMs, blocks of
grid-wide reductions) belong to a stream, or to the one launch where it is recorded into a graph; a GEMM that gets none, for
whatever reason, runs unsplit, a reduction recorded when there are no more takes its stream's."""
import re

import pytest

import dispatch
from test_gpu_dense_ragged import RAGGED, WHOLE, ragged_lengths
from test_gpu_gemm_split import DENSE_TILES, W4_TILES, W8_TILES

TICKETS = 512 * 4                                                    # bytes a stream keeps


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    folder = tmp_path_factory.mktemp("dispatch")
    return folder, dispatch.build(str(folder))


@pytest.fixture
def gpu(pkg, library, request):
    folder, path = library
    return dispatch.Dispatch(pkg, path, str(folder / (request.node.name.replace("/", "_") + ".so")))


def _calls(gpu, pkg):
    """One call of each family that splits its K."""
    return [lambda s: gpu.w8a8(s, 200, 12288, 512), lambda s: gpu.w4a16(s, 64, 8256, 96, 64), lambda s: gpu.linear(s, 100, 11520, 320, pkg.F16),
            lambda s: gpu.linear(s, 100, 11520, 320, pkg.F16, route=0, q_dtype=pkg.I8)]


def test_tickets_belong_to_a_stream_or_to_a_recorded_launch(gpu, pkg):
    calls = _calls(gpu, pkg)
    eager = {}
    for stream in (8, 16):
        words = {call(stream)[2][3] for call in calls for _ in range(2)}
        assert len(words) == 1                                       # launches of one stream follow one another
        eager[stream] = words.pop()
    assert abs(eager[8] - eager[16]) >= TICKETS
    taken = []                                                       # [first, past the last) of what was recorded
    for stream in (8, 16, 24, 8):
        gpu.capturing(stream, True)
        for call in calls:
            name, on, split = call(stream)
            assert on == stream and split[0] > 1, name
            taken.append((split[3], split[3] + 4))
        gpu.capturing(stream, False)
    # a launch's words end where the next one's begin at the latest, and none are a stream's
    taken.sort()
    assert all(a[1] <= b[0] and a[0] % 128 == 0 for a, b in zip(taken, taken[1:]))
    assert all(t[0] >= e + TICKETS or t[1] <= e for t in taken for e in eager.values())
    assert [call(8)[2][3] for call in calls] == [eager[8]] * len(calls)


@pytest.mark.parametrize("tiles_n,tiles", [(512, 8), (4096, 32), (96, 1)])
def test_a_recorded_launch_has_a_word_for_every_tile(gpu, tiles_n, tiles):
    gpu.capturing(8, True)
    first = gpu.w8a8(8, 200, 12288, tiles_n)
    second = gpu.w8a8(8, 200, 12288, tiles_n)
    assert first[2][0] > 1 and second[2][3] - first[2][3] >= 4 * tiles


def test_a_call_without_tickets_runs_unsplit(gpu, pkg):
    calls = _calls(gpu, pkg)
    split = [call(8)[2][0] for call in calls]
    assert min(split) > 1
    # the stream handle that names another stream in every thread
    assert all(call(2)[2] is None or call(2)[2][0] == 1 for call in calls)
    # more streams than the library keeps blocks for; one given back serves the next
    for stream in range(1, 256):
        assert calls[1](4096 + 8 * stream)[2][0] > 1
    for call in calls:
        name, _, s = call(64)
        assert s is None or s[0] == 1, name
    assert not gpu.lib.mtrt_hip_last_error()
    gpu.lib.fake_destroy_stream(4096 + 8)
    assert [call(64)[2][0] for call in calls] == split


def test_recorded_words_run_out_without_a_failure(gpu):
    """Nothing that was recorded is handed out again, also not after its stream is gone; what comes after them runs unsplit."""
    gpu.capturing(8, True)
    seen = set()
    while True:
        _, _, split = gpu.w8a8(8, 200, 14336, 8192)
        if split is None or split[0] == 1:
            break
        assert split[3] not in seen
        seen.add(split[3])
        assert len(seen) <= 1 << 17
    assert len(seen) == (4 << 20) // 128 and not gpu.lib.mtrt_hip_last_error()       # 128 tiles each
    gpu.capturing(8, False)
    gpu.lib.fake_destroy_stream(8)
    gpu.capturing(8, True)
    _, _, split = gpu.w8a8(8, 200, 14336, 8192)
    assert split is None or split[0] == 1
    assert gpu.w8a8(16, 200, 14336, 8192)[2][0] > 1           # eager work is not concerned


def test_a_reset_clears_what_was_recorded_on_the_stream(gpu):
    gpu.capturing(8, True)
    recorded = [gpu.w8a8(8, 200, 12288, 512)[2][3] for _ in range(3)]
    gpu.capturing(8, False)
    eager = gpu.w8a8(8, 200, 12288, 512)[2][3]
    del gpu.fills[:]
    assert gpu.lib.mtrt_hip_reset_reductions(8) == 0
    for words in recorded + [eager]:
        assert any(p <= words and words + 32 <= p + 4 * n for p, n, _ in gpu.fills), gpu.fills


def test_recorded_reductions_have_blocks_of_their_own(gpu, pkg):
    calls = [lambda s: gpu.amax(s, pkg.BF16), lambda s: gpu.dynamic(s, pkg.F32, pkg.I8)]
    eager = {stream: {call(stream)[2] for call in calls} for stream in (8, 16)}
    assert all(len(blocks) == 1 for blocks in eager.values())
    taken = []
    for stream in (8, 24, 16):
        gpu.capturing(stream, True)
        taken += [call(stream)[2] for call in calls]
        gpu.capturing(stream, False)
    every = sorted(taken + [b for blocks in eager.values() for b in blocks])
    assert all(a + 4 * 32 * 50 <= b for a, b in zip(every, every[1:]))   # 33 lines of amax.hip, 17 of dynq.hip
    assert not gpu.fills or all(stream in (8, 16) for _, _, stream in gpu.fills)
    assert {call(8)[2] for call in calls} == eager[8]
    del gpu.fills[:]
    assert gpu.lib.mtrt_hip_reset_reductions(8) == 0
    for block in taken[:2] + list(eager[8]):
        assert any(p <= block and block + 4 * 2048 <= p + 4 * n for p, n, _ in gpu.fills), gpu.fills


def test_reductions_recorded_when_the_blocks_are_gone_take_their_streams(gpu, pkg):
    gpu.capturing(8, True)
    own = [gpu.amax(8, pkg.F32)[2] for _ in range(2048)]
    assert len(set(own)) == 2048
    shared = gpu.amax(8, pkg.F32)[2]
    assert shared not in own and gpu.amax(8, pkg.F32)[2] == shared
    gpu.capturing(8, False)
    assert gpu.amax(8, pkg.F32)[2] == shared
    gpu.lib.fake_destroy_stream(8)                                   # a graph names the block: it goes to nobody else
    assert shared not in {gpu.amax(8 + 8 * k, pkg.F32)[2] for k in range(255)}


def test_last_kernel_is_the_symbol_that_was_launched(gpu, pkg):
    """Over every family and route, at sizes that take each kernel of it at some point."""
    import random
    r = random.Random(3)
    seen = set()
    for _ in range(1500):
        M, K, N = int(2 ** r.uniform(0, 12)), 128 * int(2 ** r.uniform(0, 6.5)), int(2 ** r.uniform(3, 14))
        for call in (lambda: gpu.w8a8(8, M, K, N), lambda: gpu.w8a8(8, M, K, N, scratch=False), lambda: gpu.w4a16(8, M, K, N, r.choice([64, 128])),
                     lambda: gpu.linear(8, M, K, N, pkg.F16), lambda: gpu.linear(8, M, K, N, pkg.BF16, q_dtype=pkg.F8E4M3FN),
                     lambda: gpu.linear(8, M, K, N, pkg.F16, route=0, q_dtype=pkg.I8), lambda: gpu.linear(8, M, K, N, pkg.F16, route=1)):
            name, _, split = call()
            assert gpu.lib.mtrt_hip_last_kernel().decode() == name
            seen.add((name, split is not None and split[0] > 1))
    with open(pkg.KERNEL_MODULE_PATH, "rb") as f:
        image = f.read()
    for name, _ in seen:
        assert name.encode() + b"\0" in image, name
    for family in ("w8a8_frag", "dense_frag_f16"):
        tiles = ["mtrt_gemm_%s_t%s" % (family, t) for t in ("32x128", "64x128", "128x128", "128x256", "128x384", "256x256", "256x384")]
        assert {(t, False) for t in tiles} | {(t, True) for t in tiles[:4]} <= seen


@pytest.mark.parametrize("family,shape,kernel", [
    ("w8a8", (256, 128, 128), "t32x128"), ("w8a8", (700, 256, 8200), "t128x256"), ("w8a8", (2000, 128, 16416), "t128x256"), ("w8a8", (1669, 512, 9249), "t256x384"),
    ("w8a8", (100, 256, 8209), "t64x128"), ("w8a8", (128, 4096, 1030), "t32x128"), ("w8a8", (2048, 4096, 11008), "t256x384"),
    ("w4a16", (512, 256, 384), "t32x128"), ("w4a16", (9000, 128, 64), "t128x64"), ("w4a16", (256, 4096, 11008), "t128x128"),
    ("w4a16", (4096, 4096, 11008), "t256x384"), ("w4a16", (600, 256, 8480), "t128x256"), ("w4a16", (2000, 256, 8000), "t256x256"),
    ("dense", (65, 2048, 33), "t32x128"), ("dense", (700, 1024, 8200), "t128x256"), ("dense", (999, 4096, 11008), "t128x384")])
def test_the_tile_a_shape_takes(gpu, pkg, family, shape, kernel):
    name = {"w8a8": lambda: gpu.w8a8(8, *shape), "w4a16": lambda: gpu.w4a16(8, *shape), "dense": lambda: gpu.linear(8, *shape, pkg.F16)}[family]()[0]
    assert name == {"w8a8": "mtrt_gemm_w8a8_frag_", "w4a16": "mtrt_gemm_w4a16_", "dense": "mtrt_gemm_dense_frag_f16_"}[family] + kernel


@pytest.mark.parametrize("shape,kernel", [
    ((92, 640, 6336), "t32x128"), ((1001, 896, 640), "t32x128"), ((805, 1536, 768), "t32x128x2"), ((606, 1280, 384), "t32x128"), ((579, 1152, 1550), "t32x128x2"),
    ((33, 576, 320), "t32x128"), ((300, 960, 257), "t32x128"), ((300, 960, 256), "t32x128"), ((300, 1088, 256), "t32x128x2"), ((300, 512, 2000), "t32x128"),
    ((33, 64, 64), "t32x128"), ((748, 64, 127), "t32x128"), ((512, 256, 4096), "t128x128")])
def test_few_tiles_are_not_estimated_below_what_one_of_them_takes(gpu, shape, kernel):
    """However short K is and however few the columns are."""
    assert gpu.w4a16(8, *shape, 64)[0] == "mtrt_gemm_w4a16_" + kernel


def test_a_kept_plan_is_the_calls_own(gpu, pkg):
    """Calls in an order in which each asks for another plan than the one before it, and in one in which none does, take the same launches."""
    calls = [lambda s=s, f=f, scratch=scratch: f(8, *s, scratch=scratch) for s in ((200, 12288, 512), (200, 512, 12288), (201, 12288, 512), (64, 8192, 96))
             for f in (gpu.w8a8, gpu.w4a16) for scratch in (True, False)]
    calls += [lambda s=s, dt=dt: gpu.linear(8, *s, dt) for s in ((200, 12288, 512), (100, 11520, 320)) for dt in (pkg.F16, pkg.BF16)]
    in_turn = [c() for _ in range(2) for c in calls]
    assert in_turn[:len(calls)] == in_turn[len(calls):]
    assert [c() for c in calls for _ in range(2)][1::2] == in_turn[:len(calls)]
    assert len({(name, split) for name, _, split in in_turn}) > 8


@pytest.mark.parametrize("family,tiles", [("w8a8_frag", W8_TILES), ("w4a16", W4_TILES), ("dense_frag_f16", DENSE_TILES)])
def test_the_shapes_that_test_every_tile_take_it(gpu, pkg, family, tiles):
    call = {"w8a8_frag": lambda *s: gpu.w8a8(8, *s), "w4a16": lambda *s: gpu.w4a16(8, *s, 64),
            "dense_frag_f16": lambda *s: gpu.linear(8, *s, pkg.F16)}[family]
    for shape, tile, split in tiles:
        name, _, s = call(*shape)
        assert (name, s is not None and s[0] > 1) == ("mtrt_gemm_%s_%s" % (family, tile), bool(split)), shape


@pytest.mark.parametrize("dtype,vector", [("F32", 4), ("F16", 8), ("BF16", 8)])
def test_tensors_of_64_gib_are_divided_in_64_bits(gpu, pkg, dtype, vector):
    for d0, d1 in ((1 << 16, vector << 16), (16, vector << 28), (((1 << 32) // 4099 + 16) // 16 * 16, vector * 4099)):
        for rows, far in ((d0 - 16, False), (d0, True)):
            assert (rows * (d1 // vector) >= 1 << 32) == far
            if rows:
                assert gpu.lib.mtrt_hip_nvfp4_dequantize(None, 256, 256, 256, 256, getattr(pkg, dtype), rows, d1, 0) == 0
                assert gpu.launches[-1][0] == ("mtrt_nvfp4_dqc_far_" if far else "mtrt_nvfp4_dqc_") + dtype.lower()


def test_launches_have_less_than_2_to_the_32_work_items(gpu, pkg):
    """Operands that fit into the device's 288 GB and need more workgroups of some kernels than a launch can have."""
    L = gpu.lib
    for dtype, m, k, n in ((pkg.F32, 1, 1536, (1 << 25) + 40), (pkg.F32, 1, 5, (1 << 27) - 3), (pkg.F32, 8, 1536, (1 << 25) + 1), (pkg.F32, 20, 1600, 1 << 25),
                           (pkg.F32, 32, 1537, 1 << 24), (pkg.F32, 32, 4, 1 << 29), (pkg.F32, 64, 32, (1 << 28) + 9), (pkg.F32, 120, 32, 1 << 27), (pkg.F32, 1 << 17, 32, 1 << 17),
                           (pkg.F32, 1 << 24, 32, 1000), (pkg.F16, 1, 9, (1 << 30) + 1), (pkg.BF16, 33, 200, (1 << 29) + 3), (pkg.F16, 4, 64, 1 << 28)):
        assert L.mtrt_hip_linear_dense(None, 256, 256, 256, 256, dtype, m, k, n) == 0
    for n in ((1 << 26) + 1, 1 << 27, (1 << 27) + 7):
        for q_dtype in (-1, pkg.F8E4M3FN):
            gpu.linear(8, 3, 128, n, pkg.BF16, q_dtype=q_dtype)
    assert len(gpu.sizes) > 15
    over = [(name, grid, block) for name, grid, block in gpu.sizes if grid * block >= 1 << 32]
    assert not over


@pytest.mark.parametrize("dtype,vector", [("F32", 4), ("BF16", 8)])
@pytest.mark.parametrize("vectors", [(1 << 33) - 1024, 1 << 33, (1 << 33) + 4, 3 << 33])
def test_dequantize_takes_as_many_launches_as_the_tensor_needs(gpu, pkg, dtype, vector, vectors):
    q, scales, y = 1 << 12, 1 << 44, 1 << 45
    assert gpu.lib.mtrt_hip_nvfp4_dequantize(None, q, scales, 256, y, getattr(pkg, dtype), vectors // 4, 4 * vector, 1) == 0
    assert all(grid * block < 1 << 32 and (grid - 1) * 512 < count <= grid * 512
               for (_, grid, block), (_, _, (_, _, _, count)) in zip(gpu.sizes, gpu.launches))
    done = 0
    for _, _, (q_at, s_at, y_at, count) in gpu.launches:
        assert (q_at, s_at, y_at) == (q + done * vector // 2, scales + done * vector // 16, y + done * 16) and done * vector % 16 == 0
        done += count
    assert done == vectors and (len(gpu.launches) == 1) == (vectors < 1 << 33)


@pytest.mark.parametrize("dtype,vector", [("F32", 4), ("F16", 8), ("BF16", 8)])
def test_nvfp4_quantizes_few_vectors_a_lane_of_small_and_huge_tensors(gpu, pkg, dtype, vector):
    per, cached = 256 * 256, (192 << 20) // 16             # a vector for each lane of a workgroup on each unit
    for nvec, trips in ((4, 2), (8 * per, 2), (8 * per + 4, 4), (32 * per, 4), (32 * per + 4, 8), (cached - 4, 8), (cached, 2), (1 << 32, 2), ((1 << 32) + 4, 8), (1 << 34, 8)):
        assert gpu.lib.mtrt_hip_nvfp4_quantize(None, 256, getattr(pkg, dtype), 256, 256, 256, nvec // 4, 4 * vector, 1) == 0
        name, grid, block = gpu.sizes[-1]
        assert name == "mtrt_nvfp4_q%s_%s" % ("" if trips == 8 else trips, dtype.lower()) and block == 256
        assert (grid - 1) * 256 * trips < nvec <= grid * 256 * trips and grid * block < 1 << 32


@pytest.mark.parametrize("M,N", [(4096, 2305), (3585, 4097), (9000, 1281), (4096, 2304), (4096, 2306), (2048, 11008), (5000, 65537)])
def test_large_tiles_cover_the_output(gpu, pkg, M, N):
    """256 x 256 tiles, also where the last panel holds one column; launches cut into half panels have more workgroups."""
    tiles = ((M + 255) // 256) * ((N + 255) // 256)
    assert gpu.lib.mtrt_hip_gemm_w8a8(None, 256, 256, 256, 256, 256, M, 4096, N) == 0
    assert gpu.lib.mtrt_hip_linear_dense(None, 256, 256, None, 256, pkg.F16, M, 4096, N) == 0
    assert [name for name, _, _ in gpu.sizes] == ["mtrt_gemm_w8a8_nk", "mtrt_gemm_dense_mfma_f16"]
    assert all(grid >= tiles for _, grid, _ in gpu.sizes)


@pytest.mark.parametrize("M,K,N,kernel", [(2048, 4096, 11008, "t256x128"), (4096, 4096, 4096, "t256x128"), (2048, 512, 8192, "t128x128"), (128, 256, 65536, "t128x128"),
                                          (512, 4096, 4096, "mfma"), (300, 3072, 2048, "mfma"), (1 << 19, 4096, 4096, "t128x128"), (1 << 19, 2048, 1024, "t128x128")])
def test_float32_products_take_the_tiles_that_fill_the_chip(gpu, pkg, M, K, N, kernel):
    """... of 256 x 128 only while both operands lie below 4 GiB."""
    assert gpu.lib.mtrt_hip_linear_dense(None, 256, 256, None, 256, pkg.F32, M, K, N) == 0
    assert gpu.launches[-1][0] == "mtrt_gemm_dense_%s_f32" % kernel


@pytest.mark.parametrize("M", [9, 32])
def test_up_to_32_rows_of_float32_take_every_form(gpu, pkg, M):
    """One kernel's name: 32-column tiles, or groups of eight rows on the vector units whose waves share K or take columns of their own.
    The shapes of the GPU test take all three, in launches of the workgroups that each form needs."""
    seen = set()
    for K, N in WHOLE:
        assert gpu.lib.mtrt_hip_linear_dense(None, 256, 256, None, 256, pkg.F32, M, K, N) == 0
        (name, grid, block), (_, tiles, shared) = gpu.sizes[-1], gpu.forms[-1]
        assert name == "mtrt_gemm_dense_rows32_f32"
        if tiles:
            assert (grid, block) == ((N + 31) // 32, 512)
        else:
            blocks, groups = (N + (3 if shared else 15)) // (4 if shared else 16), (M + 7) // 8
            assert block == 256 and grid % (8 * groups) == 0 and blocks <= grid // groups < blocks + 8
        seen.add("tiles" if tiles else "shared" if shared else "own")
    assert seen == {"tiles", "shared", "own"}


@pytest.mark.parametrize("dtype,item", [("F32", 4), ("F16", 2), ("BF16", 2)])
def test_rows_that_are_no_whole_slices_take_every_form(gpu, pkg, dtype, item):
    """One kernel's name: 128 x 128 tiles, 32 x 32 tiles on four waves and (float32) on eight, those only for rows of 16 bytes and more."""
    seen = set()
    for M, N in RAGGED:
        for K in ragged_lengths(item):
            assert gpu.lib.mtrt_hip_linear_dense(None, 256 + item, 256 + item, None, 256, getattr(pkg, dtype), M, K, N) == 0
            name, grid, block = gpu.sizes[-1]
            if not name.startswith("mtrt_gemm_dense_edge_"):
                continue
            waves = gpu.forms[-1][1]
            side = 32 if waves else 128
            tiles = ((M + side - 1) // side) * ((N + side - 1) // side)
            assert block == (64 * waves or 256) and (tiles <= grid < tiles + 8 if waves else grid == tiles)
            assert K * item >= 16 or not waves
            seen.add(waves)
    assert seen == ({0, 4, 8} if dtype == "F32" else {0, 4})


def test_strips_of_more_than_16_rows_cover_the_output_and_need_no_workspace(gpu):
    """Whole groups of 16 rows to a launch, at least one workgroup and at most one to a tile of columns each; on both sides of the rule's lines the
    workspace asked for is what the launch takes."""
    seen = set()
    for M in (17, 32, 33, 100, 497, 512, 513):
        for K in (128, 256, 384, 512, 896, 1024, 1408, 6272, 9216, 9344, 12288, 12416, 14336):
            for N in (1, 16, 17, 250, 500, 1000, 4000, 9000):
                for block in (64, 128):
                    name = gpu.w4a16(8, M, K, N, block)[0]
                    grid, wants = gpu.sizes[-1][1], gpu.lib.mtrt_hip_gemm_w4a16_workspace(M, K, N, block)
                    strips, groups, tiles = "strips" in name, (M + 15) // 16, (N + 15) // 16
                    each = -(-tiles // (256 // groups))              # tiles side by side, a workgroup to a unit
                    wide = M > 32
                    assert strips == (M <= 512 and (each == 1 or (each == 2 and (256 <= K <= 12288 if wide else K >= 1024)) or
                                                    (each == 3 and wide and 512 <= K <= 9216))), (M, K, N)
                    seen.add((strips, wide))
                    if strips:
                        assert grid % groups == 0 and 1 <= grid // groups <= tiles and grid <= 256 and -(-tiles // (grid // groups)) == each and wants == 0
                        assert name.endswith("_b64") == (block == 64)
                    elif wants:
                        assert gpu.launches[-1][2][0] > 1
    assert seen == {(True, True), (True, False), (False, True), (False, False)}


@pytest.mark.parametrize("family,shape,kernel", [
    ("w8a8", (3043, 768, 13632), "t128x256"), ("w8a8", (2817, 768, 5376), "t128x256"), ("w8a8", (2817, 512, 5376), "t128x256"), ("w8a8", (2643, 128, 10112), "t128x256"), ("w8a8", (2048, 512, 11008), "t256x384"), ("w8a8", (999, 4096, 11008), "t128x384"),
    ("dense", (2817, 384, 5391), "t128x256"), ("dense", (2817, 256, 5376), "t128x256"), ("dense", (3636, 64, 5824), "t128x256"), ("dense", (2981, 1472, 8768), "t256x256")])
def test_pairs_of_tiles_however_short_k_is(gpu, pkg, family, shape, kernel):
    name = gpu.w8a8(8, *shape)[0] if family == "w8a8" else gpu.linear(8, *shape, pkg.F16)[0]
    assert name == {"w8a8": "mtrt_gemm_w8a8_frag_", "dense": "mtrt_gemm_dense_frag_f16_"}[family] + kernel


def test_w8a8_of_up_to_32_rows(gpu):
    """One kernel up to 16 rows, however long K and few the columns, another up to 32: a workgroup to a tile of 32 columns, or, between one and two tiles to a
    unit, a workgroup to a unit from 9 rows on, and above 16 where K is long for the tiles left over."""
    seen = set()
    for M in (1, 8, 9, 16, 17, 32):
        for K in (128, 1920, 2048, 2688, 4096, 8192, 14336):
            for N in (1, 512, 4096, 8192, 8193, 9216, 10240, 10241, 12289, 16384, 16385):
                name = gpu.w8a8(None, M, K, N)[0]
                assert name == ("mtrt_gemm_w8a8_small16" if M <= 16 else "mtrt_gemm_w8a8_frag_rows32")
                tiles = (N + 31) // 32
                shared = 256 < tiles <= 512 and (M > 8 if M <= 16 else K >= 2048 and (tiles - 256) * 32 <= K)
                assert gpu.sizes[-1][1:] == (256 if shared else tiles, 256), (M, K, N)
                seen.add((M > 16, shared))
    assert len(seen) == 4


@pytest.mark.parametrize("M", [1, 16, 17, 25, 32])
def test_w8a8_of_few_rows_reads_some_weights_through_the_caches(gpu, M):
    """Up to 64 MiB: with half a tile to a unit at most from 8 MiB on, with more than 16 rows from 16 MiB on."""
    for K, N, few, more in ((128, 1, 1, 1), (1152, 9216, 1, 1), (4096, 2047, 1, 1), (4096, 2048, 0, 0), (14336, 512, 1, 1), (14336, 640, 0, 0), (4096, 4096, 0, 0),
                            (4096, 4097, 1, 0), (3968, 4097, 1, 1), (2048, 11008, 1, 0), (16384, 4096, 0, 0), (16512, 4096, 1, 1), (4096, 16384, 1, 0), (4096, 16385, 1, 1)):
        gpu.w8a8(None, M, K, N)
        assert gpu.forms[-1] == (("mtrt_gemm_w8a8_small16", few) if M <= 16 else ("mtrt_gemm_w8a8_frag_rows32", more)), (K, N)


def test_16_bit_linears_of_few_rows_read_weights_of_more_than_48_mib_past_the_caches(gpu, pkg):
    for N, past in ((1024, 0), (12288, 0), (12289, 1), (16384, 1)):
        gpu.linear(None, 2, 2048, N, pkg.F16)
        assert gpu.forms[-1] == ("mtrt_gemm_dense_frag_f16_rows16", past)
        gpu.linear(None, 4, 2048, N, pkg.BF16, q_dtype=pkg.F8E4M3FN)
        assert gpu.forms[-1] == ("mtrt_gemm_dense_frag_bf16_rows16_f8", past)


@pytest.mark.parametrize("dtype,item", [("F32", 4), ("F16", 2), ("BF16", 2)])
def test_softmax_rows_that_share_cache_lines_are_read_through_the_caches_from_20_to_80_mib(gpu, pkg, dtype, item):
    """... in every form of the kernel, and of rows that are whole lines none, whatever their size."""
    low, high, seen = 20 << 20, 80 << 20, set()
    for row_bytes in (20, 64, 100, 192, 400, 1000, 1040, 3000, 3008, 4112, 10004, 12016, 18004, 20016, 49016, 200000, 128, 256, 1920, 2048, 3968, 8192, 24064, 65536, 1 << 17):
        for rows, inside in ((1, False), (low // row_bytes, False), (low // row_bytes + 1, True), (high // row_bytes, True), (high // row_bytes + 1, False), ((1 << 36) // row_bytes, False)):
            assert gpu.lib.mtrt_hip_softmax(None, 256, 256, getattr(pkg, dtype), rows, row_bytes // item) == 0
            name = gpu.launches[-1][0]
            assert name.endswith("t") == (inside and row_bytes % 128 != 0), (rows, row_bytes, name)
            seen.add(name)
    forms = {re.sub("[ea]t$", "t", n.split("_")[3]) for n in seen}
    assert {f + "t" for f in ("u8v1", "u16v1", "u32v1", "u64v1", "u64v4", "v4", "v16", "g256v8", "g1024v16")} <= forms, forms


@pytest.mark.parametrize("dtype,item", [("F32", 4), ("F16", 2), ("BF16", 2)])
def test_whole_vectors_off_the_cache_lines_are_cut_from_14_mib(gpu, pkg, dtype, item):
    """By the kernels that end in c where they go past the caches; rows that start on lines by none."""
    for row_bytes, form in ((528, "v1"), (1040, "v2"), (2064, "v4"), (6000, "v8"), (10000, "v16"), (1024, None), (3968, None)):
        at = -(-(14 << 20) // row_bytes)                             # the least number of rows of 14 MiB
        for x, rows in [(x, rows) for x in (256, 256 + 16, 256 + 128) for rows in (1, at - 1, at, (20 << 20) // row_bytes, (80 << 20) // row_bytes + 1)]:
            assert gpu.lib.mtrt_hip_softmax(None, x, 256, getattr(pkg, dtype), rows, row_bytes // item) == 0
            name = gpu.launches[-1][0]
            off = row_bytes % 128 != 0 or x % 128 != 0
            assert name.endswith("c") == (off and rows >= at), (x, row_bytes, rows, name)
            assert not form or name.split("_")[3] == form + ("c" if rows >= at else ""), name
