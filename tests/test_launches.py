"""What calls launch, in what order and with how much scratch: the library on a stand-in for the HIP runtime (tests/cpp), and the
same between two threads on the GPU."""
import os
import subprocess
import threading

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def on_stand_in(tmp_path, name, lines=""):
    import awesome_fusion_amd as af
    lib, exe = os.path.dirname(af.library_path()), str(tmp_path / name)
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-rdynamic", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "cpp", name + ".cc"), "-o", exe, "-L" + lib, "-l:libbfaintb_gemm.so",
                    "-Wl,-rpath," + lib, "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib", "-lpthread"], check=True)
    return subprocess.run([exe], input=lines, capture_output=True, text=True, timeout=60)


def calls(tmp_path, lines):
    """(return code, launches, workgroups of the first launch) of each call: "m n k weight_bits kind workspace_bytes"."""
    r = on_stand_in(tmp_path, "call_launches", "\n".join(lines))
    assert r.returncode == 0
    return [tuple(map(int, line.split())) for line in r.stdout.split("\n") if line]


def test_launches_of_one_call_follow_one_another(tmp_path):
    r = on_stand_in(tmp_path, "test_launch_order")
    assert r.returncode == 0 and "all checks passed" in r.stdout, r.stdout[-3000:]


# (shape, code width, packed, bytes without a second launch: what these calls needed before there was one)
SCRATCH = [((124, 2800, 1664), 8, 0, 0), ((235, 1168, 1792), 8, 0, 0), ((105, 4560, 3200), 8, 1, 0), ((96, 4096, 11008), 8, 0, 4718848),
           ((96, 4112, 7296), 4, 1, 3158272), ((33, 3200, 4608), 4, 0, 1689856), ((474, 1136, 1920), 8, 0, 0), ((991, 4832, 11392), 4, 0, 0),
           ((1522, 2784, 8448), 8, 1, 0), ((314, 1120, 12672), 8, 1, 5627136), ((1, 4096, 4096), 8, 0, 114944)]


def test_less_scratch_than_the_plan_needs(tmp_path):
    """A caller who brings less than a second launch needs gets the product without one, if it fits, in one launch (or two
    that share nothing); who brings less than that is refused."""
    import awesome_fusion_amd as af
    asked, wants = [], []
    for (m, n, k), bits, packed, least in SCRATCH:
        full = (af.prepacked_workspace_bytes if packed else af.workspace_bytes)(m, n, k, bits)
        launches = af.plan(m, n, k, bits, packed=packed).launches
        assert full > least or launches == 1
        for nbytes, want in ((full, (0, launches)), (full - 256, (0, 1) if full > least else (-6, 0)), (least, (0, 1)), (least - 256, (-6, 0))):
            if nbytes >= 0:
                asked.append(f"{m} {n} {k} {bits} {packed} {nbytes}")
                wants.append(want)
    got = [x[:2] for x in calls(tmp_path, asked)]
    assert got == wants, [x for x in zip(asked, got, wants) if x[1] != x[2]]


def test_a_first_call_under_capture_needs_no_second_launch(tmp_path):
    """bfaintb_gemm_static before the device is set up, under capture: shapes that need its scratch for a second launch only are
    served without one; a shape for the decode kernels, which need the set-up, is refused."""
    shapes = [(63, 4784, 1368), (54, 4160, 1328), (96, 4096, 11008), (4096, 4096, 4096)]
    assert [x[:2] for x in calls(tmp_path, ["%d %d %d 8 2 0" % s for s in shapes])] == [(0, 1), (0, 1), (-8, 0), (0, 1)]


def test_reference_arithmetic_takes_the_kernel_it_has(tmp_path):
    """The reference's arithmetic has no tiles with k split: where only those lead the decode family, it gets the family, with
    the scratch that bfaintb_gemm_workspace_bytes asks for; without scratch it gets the tiles, unsplit."""
    import awesome_fusion_amd as af
    for shape in ((96, 4096, 11008), (64, 4096, 11008), (124, 2800, 1664), (300, 1040, 8192)):
        assert af.variant(*shape) == af.PREFILL
        family = af.plan(*shape, which=af.DECODE)
        line = "%d %d %d 8 3 " % shape
        (rc, launches, workgroups), bare = calls(tmp_path, [line + str(af.workspace_bytes(*shape)), line + "0"])
        assert (rc, launches, workgroups) == (0, 1, family.workgroups), (shape, workgroups, family.workgroups)
        assert bare[:2] == (0, 1) and (family.splits == 1 or bare[2] < workgroups)


# (shape, code width, group, packed, tile rows): the family, the slab kernel, every height of tiles with and without the copying wave, split k in
# one launch and in two, the large tiles and their thin last round, a product in two launches by rows
PLANS = [((1, 4096, 4096), 8, 0, 0, 16), ((8, 4096, 4096), 4, 128, 1, 16), ((32, 4096, 4096), 8, 0, 1, 16), ((40, 4096, 4096), 8, 0, 0, None),
         ((17, 22016, 2048), 8, 0, 0, 32), ((32, 22016, 4096), 4, 128, 0, 32), ((32, 22016, 4096), 4, 128, 1, 32), ((20, 20480, 4096), 8, 0, 1, 32),
         ((96, 4096, 11008), 8, 0, 0, 96), ((64, 20480, 4096), 4, 128, 1, 64), ((96, 36864, 8192), 8, 0, 0, 96), ((128, 20480, 4096), 8, 64, 1, 128),
         ((48, 18432, 8192), 8, 0, 0, 64), ((640, 4096, 4096), 8, 64, 0, 128), ((785, 1440, 4480), 8, 32, 0, 128), ((320, 16384, 4096), 8, 0, 0, 160),
         ((384, 16384, 4096), 4, 128, 1, 192), ((512, 11008, 4096), 8, 0, 0, 256), ((512, 11008, 512), 8, 0, 0, 256), ((4096, 4096, 4096), 8, 0, 0, 256),
         ((2048, 28672, 8192), 4, 128, 0, 256), ((577, 13824, 5120), 4, 128, 1, None)]


def test_the_plan_describes_what_is_launched(tmp_path):
    """Rows of a tile, waves, workgroups (the tiled kernels launch a whole number of them per XCD, an eighth each) and launches; and the same
    for every variant by name."""
    import awesome_fusion_amd as af
    asked = [(s, b, g, pk, rows, v) for s, b, g, pk, rows in PLANS
             for v in (af.AUTO, af.DECODE, af.PREFILL, af.PREFILL_128, af.PREFILL_256, af.PREFILL_256X128, af.PREFILL_128_LDS, af.PREFILL_256_LDS)]
    r = on_stand_in(tmp_path, "plan_launches", "\n".join("%d %d %d %d %d %d %d 0" % (*s, b, g, pk, v) for s, b, g, pk, _, v in asked))
    assert r.returncode == 0
    answers = [tuple(map(int, line.split())) for line in r.stdout.split("\n") if line]
    assert len(answers) == len(asked)
    kinds = set()
    for q, (variant, kernel, rows, cols, waves, splits, wgs, tail, launches, rc, did, did_waves, did_wgs, did_others) in zip(asked, answers):
        (m, n, k), bits, group, packed, want, which = q
        what = (q, rows, cols, waves, splits, wgs, tail, launches, did, did_waves, did_wgs, did_others)
        assert (rc, did, did_waves) == (0, launches, waves), what
        first = wgs or tail   # (fewer large tiles than half a round are all cut in halves: the thin round is all there is)
        assert first <= did_wgs < first + 8 * splits, what
        assert which != af.AUTO or want is None or rows == want, what
        two_by_rows = which == af.AUTO and tail and kernel not in (af.KERNEL_TILES_256, af.KERNEL_TILES_256_LDS)
        if not (two_by_rows or kernel in (af.KERNEL_TILES_256, af.KERNEL_TILES_256_LDS)):
            assert wgs == -(-m // rows) * -(-n // cols) * splits, what
        assert tail <= did_others or wgs == 0, what
        kinds.add((kernel, rows))
    assert {(af.KERNEL_TILES_128, r) for r in (32, 64, 96, 128, 160, 192, 256)} <= kinds and (af.KERNEL_TILES_256X128, 256) in kinds


def test_few_rows_choose_by_the_calls_own_distance_of_rows(tmp_path):
    """17 to 32 rows over codes in rows: rows a multiple of 1024 codes apart get the family's launch, whatever n; others the tiles'."""
    import awesome_fusion_amd as af
    asked, wants = [], []
    for m, n, k, bits, group in ((17, 22016, 2048, 8, 0), (32, 22016, 4096, 8, 128), (32, 22528, 4096, 8, 0), (32, 22016, 4096, 4, 128), (20, 22016, 4096, 4, 128)):
        family, tiles = af.plan(m, n, k, bits, group, which=af.DECODE), (n + 127) // 128
        for ldb in (0, n + 16, n + 128, n // 1024 * 1024 + 1024, 32768):
            pitch = ldb or n   # (up to 20 rows of 4-bit codes: only where rows are not whole lines)
            on_tiles = pitch % 1024 != 0 and (bits == 8 or m > 20 or pitch % 256 != 0)
            asked.append("%d %d %d %d %d 0 0 %d" % (m, n, k, bits, group, ldb))
            wants.append((9, (tiles + 7) // 8 * 8) if on_tiles else (family.waves, family.workgroups))
    r = on_stand_in(tmp_path, "plan_launches", "\n".join(asked))
    assert r.returncode == 0
    got = [tuple(int(x) for x in line.split()[11:13]) for line in r.stdout.split("\n") if line]
    assert got == wants, [x for x in zip(asked, got, wants) if x[1] != x[2]]


@pytest.mark.gpu
def test_two_threads_share_a_stream():
    """The operators' workspace is one per stream: products in two launches and split decode calls from two threads."""
    import torch
    import awesome_fusion_amd as af
    import awesome_fusion_amd.torch_op as top
    torch.manual_seed(11)
    shapes = [(96, 4096, 11008), (1, 4096, 4096)]
    assert af.plan(*shapes[0]).launches == 2 and af.plan(*shapes[1]).splits > 1
    layers = [top.QuantLinear.from_float(torch.nn.Linear(k, n, bias=False).cuda(), 8, 0) for _, n, k in shapes]
    xs = [torch.randn((m, k), device="cuda", dtype=torch.bfloat16) for m, _, k in shapes]
    want = [layer(x) for layer, x in zip(layers, xs)]
    torch.cuda.synchronize()
    outs = [[], []]

    def work(i):
        for rep in range(40):
            j = (rep + i) % 2
            outs[i].append((j, layers[j](xs[j])))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert all(len(o) == 40 for o in outs)
    assert all(torch.equal(c, want[j]) for o in outs for j, c in o)


# shapes (width of the codes last) that the slab kernel, which needs neither scratch nor the device's set-up, served before the family had fewer than
# eight column blocks a workgroup: those the family leads now, unsplit, and those it would lead if it did not split k
NOW_FAMILY = [(5, 42576, 10752, 4), (7, 19216, 14336, 4), (13, 33872, 8320, 8), (11, 18992, 3200, 8), (6, 22144, 2048, 4)]
STILL_SLAB = [(5, 1456, 6912, 8), (2, 10576, 1408, 4), (13, 3056, 6400, 8), (3, 13776, 2176, 4)]


def test_calls_of_the_slab_kernel_need_no_scratch_and_no_set_up(tmp_path):
    import awesome_fusion_amd as af
    for m, n, k, bits in NOW_FAMILY:
        pl = af.plan(m, n, k, bits, packed=True)
        assert (pl.kernel, pl.splits, pl.workspace_bytes) == (af.KERNEL_DECODE_FAMILY, 1, 0), pl.as_dict()
    for m, n, k, bits in STILL_SLAB:
        assert af.plan(m, n, k, bits, packed=True).kernel == af.KERNEL_DECODE_SLAB
    shapes = NOW_FAMILY + STILL_SLAB
    slabs = [(0, 1, n // 16 * -(-m // 32)) for m, n, _, _ in shapes]
    r = on_stand_in(tmp_path, "packed_first_capture", "\n".join("%d %d %d %d" % s for s in shapes))
    assert r.returncode == 0
    assert [tuple(map(int, line.split())) for line in r.stdout.split("\n") if line] == slabs
    got = calls(tmp_path, ["%d %d %d %d 1 0" % s for s in shapes])
    assert [x[:2] for x in got] == [(0, 1)] * len(shapes)
    assert [x[2] for x in got[:len(NOW_FAMILY)]] == [af.plan(m, n, k, bits, packed=True).workgroups for m, n, k, bits in NOW_FAMILY]


# many rows and a short k (width of the codes last): tiles, which need neither scratch nor the device's set-up
SHORT_K = [(1901, 12544, 128, 4), (516, 37184, 128, 8), (141, 43360, 256, 4), (2889, 28096, 128, 8), (350, 33264, 128, 8), (529, 25456, 256, 8), (2571, 45456, 128, 4)]


def test_a_short_k_runs_tiles_and_may_be_a_first_call_under_capture(tmp_path):
    import awesome_fusion_amd as af
    for m, n, k, bits in SHORT_K:
        for packed in (False, True):
            pl = af.plan(m, n, k, bits, packed=packed)
            assert pl.kernel >= af.KERNEL_TILES_128 and pl.splits == 1 and pl.workspace_bytes == 0, pl.as_dict()
    got = calls(tmp_path, ["%d %d %d %d %d 0" % (*s, kind) for s in SHORT_K for kind in (4, 5, 2)])
    assert [x[0] for x in got] == [0] * len(got) and all(x[1] >= 1 for x in got), got


# what tall tiles of one chain and the family's workgroups take to start, left out, made two launches of these (width of the codes, group size, packed)
NOT_TWO_LAUNCHES = [(2515, 7584, 384, 4, 128, False), (1995, 10832, 256, 8, 64, True), (564, 25648, 128, 8, 64, False), (1488, 13584, 256, 8, 32, True),
                    (2857, 12832, 128, 8, 32, True), (1130, 45424, 512, 4, 32, True), (1818, 27856, 128, 8, 64, True)]


@pytest.mark.parametrize("m,n,k,bits,group,packed", NOT_TWO_LAUNCHES)
def test_a_short_k_is_one_launch_where_two_take_longer(m, n, k, bits, group, packed):
    import awesome_fusion_amd as af
    pl = af.plan(m, n, k, bits, group, packed=packed)
    assert (pl.kernel, pl.tile_cols, pl.launches) == (af.KERNEL_TILES_256, 256, 1), pl.as_dict()


def test_a_known_call_on_tiles_of_256_columns_takes_the_host_no_longer(tmp_path):
    """The choice of these tiles is made once for a shape, not several times a call: against tall tiles, which are not asked about."""
    import awesome_fusion_amd as af
    assert af.plan(1024, 8192, 4096).kernel == af.KERNEL_TILES_128
    shapes = ["128 43680 4096 8 0", "913 9296 3328 8 1", "384 22016 4096 4 0"]
    r = on_stand_in(tmp_path, "host_time", "\n".join(["1024 8192 4096 8 0"] + shapes))
    assert r.returncode == 0
    tall, *wide = map(float, r.stdout.split())
    assert max(wide) < 1.5 * tall, (tall, wide)


# 97 to 128 rows against more than a round of small tiles: tiles of 256 columns, but where the call names a split of k, which only the small ones have
@pytest.mark.parametrize("m,n,k,bits", [(101, 38464, 3712, 4), (126, 39888, 1024, 8), (128, 43680, 4096, 8)])
def test_a_named_split_of_k_keeps_the_tiles_that_have_it(m, n, k, bits):
    import awesome_fusion_amd as af
    for which in (af.AUTO, af.PREFILL):
        assert af.plan(m, n, k, bits, which=which).tile_cols == 256
        for split in (1, 2, 3):
            pl = af.plan(m, n, k, bits, which=which, force_split_k=split)
            assert (pl.kernel, pl.tile_cols, pl.splits) == (af.KERNEL_TILES_128, 128, split), pl.as_dict()
            assert pl.workspace_bytes == af.workspace_bytes(m, n, k, bits, which=which, force_split_k=split) and (pl.workspace_bytes != 0) == (split > 1)
