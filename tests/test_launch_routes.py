"""Which kernels a call launches, in which order and on whose behalf, checked
without a GPU: the library's host code runs on a stand-in for the HIP runtime
that records launches (launch_recorder.py)."""
import pytest

import launch_recorder


@pytest.fixture(scope="module")
def recorder(tmp_path_factory):
    return launch_recorder.build(tmp_path_factory.mktemp("recorder"))


@pytest.mark.parametrize("stream", [0, 0x5000])
@pytest.mark.parametrize("one,other", [("attention(s)", "gemm(128, 1536, 8960, s)"),
                                       ("gemm(128, 1536, 8960, s, True)", "attention(s)"),
                                       ("gemm_w4a8(300, 1536, 8960, s)", "gemm_w4a8(200, 1536, 8960, s)"),
                                       ("gemm_noalloc(128, 1536, 8960, s)", "gemm_noalloc(64, 1536, 8960, s)")])
def test_partials_and_their_sum_stay_together(recorder, one, other, stream):
    """Threads that share a stream (the null stream is every thread's default)
    share its workspace: a launch's partials and the kernel that sums them are
    enqueued with nothing of another thread's in between."""
    launch_recorder.run(recorder, f"""
        s = {stream}
        reserve(s)
        R.recorder_reset(2000)
        go = threading.Barrier(3)
        def work(k):
            go.wait()
            for i in range(4):
                if k == 2: {one}
                else: {other}
        threads = [threading.Thread(target=work, args=(k,)) for k in range(3)]
        [t.start() for t in threads]
        [t.join() for t in threads]
        e = events()
        assert len(e) == 24, e  # every call here is split: two launches
        for a, b in zip(e[::2], e[1::2]):
            assert a.thread == b.thread, (a, b)
            assert ("reduce" in b.kernel or "combine" in b.kernel) and a.stream == b.stream == s, (a, b)
    """)


def test_streams_do_not_wait_for_each_other_and_release_waits_for_a_launch(recorder):
    """While one stream's launch is being enqueued, launches on another go on; a
    workspace is given up only after the launch that uses it is enqueued whole."""
    launch_recorder.run(recorder, """
        a, b = 0x5000, 0x6000
        reserve(a), reserve(b)
        R.recorder_reset(0)
        R.recorder_close(a)
        t = threading.Thread(target=gemm, args=(128, 1536, 8960, a))
        t.start()
        while R.recorder_waiting() == 0:
            time.sleep(0.001)
        gemm(128, 1536, 8960, b)  # not held up by a's launch
        r = threading.Thread(target=release, args=(a,))
        r.start()
        time.sleep(0.05)
        assert r.is_alive() and not any(e.what == "free" for e in events())
        R.recorder_open()
        t.join(), r.join()
        e = events()
        assert [x.what for x in e] == ["launch"] * 4 + ["free"], e
        assert [x.stream for x in e[:4]] == [a, b, b, a], e
        gemm(128, 1536, 8960, a)  # unsplit now
        assert len(events()) == 6
        for i in range(63):  # freed entries serve other streams: at most 64 hold one
            reserve(0x10000 + 16 * i)
        assert L.qe_gemm_reserve_workspace(V(0x90000)) == 2
        release(b)
        reserve(0x90000)
    """)


def test_recorded_prefill_attention_takes_no_workspace(recorder):
    """A graph may be replayed on any stream and after the capturing stream's
    workspace is released, so a launch recorded into one is a single kernel."""
    launch_recorder.run(recorder, """
        s = 0x5000
        reserve(s)
        attention(s)
        R.recorder_set_capturing(s, 1)
        attention(s)
        R.recorder_set_capturing(s, 0)
        attention(s)
        split, combine, one, split2, combine2 = events()
        assert "combine" in combine.kernel and (split, combine) == (split2, combine2)
        assert one.kernel == split.kernel and one.grid[0] * 10 == split.grid[0], (one, split)
    """)


def test_two_key_groups_are_never_split(recorder):
    """More blocks than CUs: two key groups a block, one kernel, whatever the
    context and the workspace; with half as many one group, split in three (what
    the workspace holds)."""
    launch_recorder.run(recorder, """
        reserve()
        for rows, blocks in ((1370, 257), (3002, 563), (680, 128)):
            for max_seq in (1024, 4096, 32768):
                R.recorder_reset(0)
                attention(0, rows, 24, 1, max_seq)
                e = events()
                if blocks > 256:
                    assert len(e) == 1 and e[0].block == 512 and e[0].grid == (blocks, 1, 1), e
                else:
                    assert len(e) == 2 and e[0].block == 256 and e[0].grid == (3 * blocks, 1, 1), e
    """)


@pytest.mark.parametrize("tiled", [False, True])
def test_forced_tile_takes_the_slices_of_its_own_family(recorder, tiled):
    """With gemm_tile 1..4 and no slice count forced, a launch runs what
    qe_gemm_prefill_plan reports, also where another kernel (few rows, LDS ring)
    would have been chosen and would have run unsplit."""
    launch_recorder.run(recorder, f"""
        tiled = {tiled}
        reserve()
        seen = set()
        for tile, (bm, bn) in enumerate([(64, 64), (64, 128), (128, 64), (128, 128)], 1):
            tune("gemm_tile", tile)
            for M in (1, 9, 32, 33, 128, 200, 700, 1024, 1500, 2048):
                for N, K in ((2048, 1536), (1536, 1536), (17920, 1536), (1536, 8960)):
                    t, s = I(), I()
                    ok(L.qe_gemm_prefill_plan(I(M), I(N), I(K), I(tiled), ctypes.byref(t), ctypes.byref(s)))
                    R.recorder_reset(0)
                    gemm(M, N, K, 0, tiled)
                    e = events()[0]
                    assert t.value == tile and e.grid == ((N + bn - 1) // bn, (M + bm - 1) // bm, s.value), (M, N, K, e)
                    assert "ILi%dELi%dE" % (bm, bn) in e.kernel, e
                    seen.add((tile, M, N, K, s.value))
        assert (1, 9, 1536, 8960, 6) in seen and (4, 2048, 1536, 8960, 1) in seen, sorted(seen)
    """)


# (rows, columns) of a block, by gemm_tile number
TILES = {1: (64, 64), 2: (64, 128), 3: (128, 64), 4: (128, 128), 5: (128, 256), 6: (128, 256), 7: (128, 128)}


@pytest.mark.parametrize("setting", ["", "gemm_staged 1", "gemm_tile 6", "gemm_tile 8", "gemm_slices 3"])
@pytest.mark.parametrize("tiled", [False, True])
def test_launch_plan_names_the_kernel_that_runs(recorder, tiled, setting):
    """qe_gemm_prefill_launch_plan against the launches made: kernel, tile and
    slices, over shapes at which the planner takes every kernel it has."""
    launch_recorder.run(recorder, f"""
        tiled, setting, TILES = {tiled}, {setting!r}.split(), {TILES}
        reserve()
        if setting:
            tune(setting[0], int(setting[1]))
        picked = set()
        for M in (1, 9, 32, 33, 64, 65, 128, 300, 512, 1000, 1024, 1500, 2048, 4096):
            for N, K in ((2048, 1536), (1536, 1536), (17920, 1536), (1536, 8960), (43, 768)):
                t, s = I(), I()
                ok(L.qe_gemm_prefill_launch_plan(I(M), I(N), I(K), I(tiled), ctypes.byref(t), ctypes.byref(s)))
                tile, slices = t.value, s.value
                R.recorder_reset(0)
                gemm(M, N, K, 0, tiled)
                e = events()
                picked.add(tile)
                assert len(e) == (1 if slices == 1 else 2), (M, N, K, e)
                name, grid = e[0].kernel, e[0].grid
                if tile == 8:
                    assert "skinny" in name and slices == 1, e
                    continue
                bm, bn = TILES[tile]
                rows, cols = (M + bm - 1) // bm, (N + bn - 1) // bn
                assert "ILi%dELi%dE" % (bm, bn) in name, (tile, e)
                if tile >= 5:
                    assert "_dma_" in name and grid == (rows * cols, slices, 1), (tile, e)
                    assert e[0].block == (256 if tile == 5 else 512), (tile, e)
                else:
                    assert ("_mfma_" in name or "_ks2_" in name) and grid == (cols, rows, slices), (tile, e)
        if not setting:
            assert picked >= (set((1, 2, 5, 6, 7, 8)) if tiled else set((1, 2, 8))), picked
        if setting == ["gemm_staged", "1"]:
            assert max(picked) <= 4, picked
    """)


def test_automatic_plans_leave_the_ring_where_it_is_slower(recorder):
    """Sides of the rule that admits an LDS-ring kernel to an automatic plan; a
    forced tile is not asked."""
    launch_recorder.run(recorder, """
        reserve()
        def kernel(M, N, K):
            t, s = I(), I()
            ok(L.qe_gemm_prefill_launch_plan(I(M), I(N), I(K), I(1), ctypes.byref(t), ctypes.byref(s)))
            R.recorder_reset(0)
            gemm(M, N, K, 0, True)
            assert ("_dma_" in events()[0].kernel) == (t.value in (5, 6, 7)), (M, N, K, t.value)
            return t.value
        for M, N, K, ring in ((72, 17920, 2048, 0), (128, 17920, 1536, 0), (256, 17920, 1536, 0),  # too few blocks
                              (384, 17920, 1536, 6), (700, 17920, 1536, 5), (1024, 17920, 1536, 5), (4096, 17920, 1536, 5),
                              (850, 12288, 1536, 0), (1200, 12288, 1536, 5),  # up to 1.5 blocks a CU, above it
                              (512, 17920, 2048, 0), (700, 12288, 2048, 0),   # more than a round of two-group blocks
                              (512, 1536, 4096, 0), (700, 1024, 4096, 0),     # 128x128 split
                              (1200, 2048, 4096, 0), (1400, 1536, 6144, 6),   # 128x256 split, short and long
                              (1200, 2048, 1536, 0), (2048, 2048, 1536, 7)):  # 128x128, rows
            got = kernel(M, N, K)
            assert got == ring if ring else got <= 4, (M, N, K, got, ring)
        for tile in (5, 6, 7):
            tune("gemm_tile", tile)
            assert kernel(128, 17920, 1536) == tile
    """)


def test_w4a8_rows_per_block(recorder):
    """Sides of the W4A8 tile rule: 128 rows a block where 128-row tiles fill 7/8 to
    all of a round, or from 9/8 of one on, or few tiles have a long K."""
    launch_recorder.run(recorder, """
        reserve()
        for M, N, K, rows in ((300, 17920, 1536, 64), (700, 8192, 1024, 64), (850, 8192, 1024, 128),
                              (1024, 8192, 1024, 128), (512, 17920, 1536, 64), (640, 14336, 1536, 64),
                              (600, 17920, 1536, 128), (1500, 17920, 1536, 128), (300, 1536, 8960, 64),
                              (1024, 1536, 8960, 128)):
            R.recorder_reset(0)
            gemm_w4a8(M, N, K)
            e = events()[0]
            assert ("ILi%dE" % rows) in e.kernel and e.grid[1] == (M + rows - 1) // rows, (M, N, K, e)
    """)


@pytest.mark.parametrize("tile", [0, 5, 6, 7])
def test_tiled_scales_at_an_odd_half_take_the_staged_kernels(recorder, tile):
    """Tiled scales need 2-byte alignment only. The LDS-ring kernels fetch them in
    4-byte pieces and are not chosen, nor forced, for others."""
    launch_recorder.run(recorder, f"""
        tune("gemm_tile", {tile})
        for M in (1024, 2048, 4096):
            R.recorder_reset(0)
            gemm(M, 17920, 1536, 0, True)
            gemm(M, 17920, 1536, 0, True, P + 2)
            gemm(M, 17920, 1536, 0, True, P + 4)
            a, b, c = events()
            assert "_dma_" in a.kernel and a[2:] == c[2:], (a, c)
            assert "_mfma_" in b.kernel or "_ks2_" in b.kernel, b
        class View(ctypes.Structure):
            _fields_ = [(n, V) for n in ("qw", "qs", "q", "kw", "ks", "k", "vw", "vs", "v")]
        for odd in ("qs", "ks", "vs"):
            R.recorder_reset(0)
            for shift in (0, 2):
                v = View(*[P] * 9)
                setattr(v, odd, P + shift)
                ok(L.qe_launch_gemm_prefill_qkv_w4a16_tiled(ctypes.byref(v), V(P), I(2048), V(0), I(1536), I(12), I(2),
                                                            I(128)))
            ring, staged = events()
            assert "_dma_" in ring.kernel and "_dma_" not in staged.kernel, (ring, staged)
    """)
