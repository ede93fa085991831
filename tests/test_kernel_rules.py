"""The host-side rules that pick a kernel and its grid for the products: pure arithmetic on the shape. What is held
here is what must stay true under any tuning (limits the kernels rely on, no dependence on the number of rows), not
the tuned numbers themselves."""
from jllm_serve_amd.kernels import ops

SHAPES = {  # (N, K, gated): qkv, o, gate/up, down
    "8b": ((6144, 4096, False), (4096, 4096, False), (12288, 4096, True), (4096, 12288, False)),
    "14b": ((7168, 5120, False), (5120, 5120, False), (17408, 5120, True), (5120, 17408, False)),
    "32b": ((10240, 5120, False), (5120, 8192, False), (25600, 5120, True), (5120, 25600, False)),
}


def test_k_parts_fill_the_rounds():
    """Whatever the tuning: every part keeps the minimum length, a part's blocks give back the count, the chosen count never
    leaves the busiest compute unit with a larger share of the product than no cut at all would, and the choice is the
    cheapest by the estimate over every number of weight rows and every count of parts that the kernel can do."""
    cus = ops.compute_units()
    shapes = [s for v in SHAPES.values() for s in v] + [(96, 128, False), (256, 256, False), (384, 1024, True), (5120, 640, False),
                                                       (1024, 3072, False), (4608, 3584, False), (18944, 3584, True), (6144, 2048, True)]
    for n, k, gated in shapes:
        rows, parts = ops._stream_plan(n, k, gated)
        nblk = k // 128
        per = -(-nblk // parts)
        assert parts >= 1 and (parts == 1 or per >= ops.STREAM_MIN_BLOCKS), (n, k, gated, parts)
        assert -(-nblk // per) == parts, (n, k, gated, parts)
        tiles = -(-n // (rows // 2 if gated else rows))
        share = lambda p: -(-(tiles * p) // cus) / (tiles * p)
        assert share(parts) <= share(1) + 1e-12, (n, k, gated, parts)
        cheapest = min(ops._stream_ns(n, k, gated, r, p) for r in (32, 64, 96, 128) for p in range(1, ops.STREAM_MOST_PARTS + 1)
                       if p == 1 or (-(-nblk // p) >= ops.STREAM_MIN_BLOCKS and -(-nblk // -(-nblk // p)) == p and
                                     -(-n // (r // 2 if gated else r)) <= ops.STREAM_COUNTERS))
        assert ops._stream_ns(n, k, gated, rows, parts) == cheapest, (n, k, gated)
    assert ops._stream_plan(151936, 4096, False)[1] == 1, "many column tiles: no cut"


def test_k_parts_do_not_depend_on_rows():
    """The rule has no argument for the number of rows: a row's sum is the same bits in any batch."""
    import inspect
    assert list(inspect.signature(ops._stream_plan.__wrapped__).parameters) == ["N", "K", "gated"]


def test_kernel_for_few_rows(monkeypatch):
    """Products of up to 16 rows go to one kernel whatever their shape (cutting K over workgroups was slower at every one that
    was measured, a launch for its counters aside), and have no scratch; those of 17 to 64 rows to the other."""
    import torch

    import recorded
    seen = recorded.record(monkeypatch)
    shapes = [(n, k) for v in SHAPES.values() for n, k, _ in v] + [(128, 512), (1024, 8192), (1280, 8192), (1024, 16384), (256, 32768)]
    for n, k in shapes:
        for rows in (1, 8, 16, 17, 64):
            a, w, res = recorded.tensor(rows, k), recorded.tensor(n, k), recorded.tensor(rows, n, dtype=torch.float32)
            del seen[:]
            promise = ops.gemm_add_then_norm(a, w, res, recorded.tensor(n), 1e-5, torch.bfloat16)
            ops.gemm(promise, recorded.tensor(512, n))
            ops.gemm(a, w)
            few = rows <= 16
            assert [name for name, _ in seen] == (["jllm_gemm_skinny_norm_bf16"] * 2 + ["jllm_gemm_skinny_bf16"] if few else ["jllm_gemm_stream_bf16"] * 3), (n, k, rows)


def test_rows_of_a_workgroup_of_the_first_weight_streaming_kernel():
    """Whatever the tuning: the extra rows divide N together with the 16, the gated product never has any (its second
    tile is the up weight), the rule knows nothing of the number of rows, and it only ever raises the share of the
    compute units' rounds that the workgroups fill."""
    import inspect
    assert list(inspect.signature(ops._skinny_second_rows.__wrapped__).parameters) == ["N", "gated"]
    for n in list(range(16, 12288 + 1, 16)) + [151936]:
        rows = ops._skinny_second_rows(n, False)
        assert rows in (0, 4, 8, 12, 16) and n % (16 + rows) == 0, (n, rows)
        assert rows == 0 or ops._round_fill(n // (16 + rows)) > ops._round_fill(n // 16), (n, rows)
        assert ops._skinny_second_rows(n, True) == 0
    assert ops._skinny_second_rows(4096, False) == 0, "N / 16 fills the compute units exactly"
    assert ops._skinny_second_rows(100, False) == 0, "an N the kernel does not take"


def test_k_splits_of_the_tiled_kernel():
    """A cut divides the K steps evenly and leaves every workgroup at least four of them; more rows never mean more
    cuts; the gated product is never cut."""
    assert ops._k_splits(128, 4096, 4096, True) == 1, "the gated epilogue needs both whole sums"
    for n, k in ((6144, 4096), (4096, 4096), (4096, 12288), (5120, 17408), (96, 128), (130, 192), (384, 4096), (192, 136 * 64)):
        last = None
        for rows in (70, 96, 128, 192, 256, 384, 512, 1000, 1024, 2048, 8192):
            s = ops._k_splits(rows, n, k, False)
            assert s >= 1 and (k // 64) % s == 0 and (s == 1 or k // 64 // s >= 4), (rows, n, k, s)
            assert last is None or s <= last, (rows, n, k, s, last)
            last = s
    assert ops._k_splits(8192, 4096, 4096, False) == 1, "enough tiles: no cut"


def test_plan_of_the_two_group_kernel():
    """Whatever the constants of its estimate: the plan names a tile the kernel has (256 rows) or none, a cut divides
    the K stages evenly and leaves every workgroup a range of the minimum length, the gated product is never cut,
    products of a few rows and shapes the kernel cannot take stay with the other kernel, and a product whose tiles
    fill the compute units many times over takes the large tile with K whole."""
    for shapes in SHAPES.values():
        for n, k, gated in shapes:
            for rows in (1, 64, 65, 128, 256, 257, 320, 448, 512, 1000, 1536, 1792, 2048, 3000, 4096, 8192):
                tile, cut = ops._pingpong_plan(rows, n, k, gated)
                assert tile in (0, 256) and cut in (1, 2, 4), (rows, n, k, gated, tile, cut)
                assert tile or cut == 1, "no tile, no cut"
                if cut > 1:
                    assert not gated and k % 64 == 0 and (k // 32) % cut == 0 and k // cut >= ops.PINGPONG_SPLIT_MIN_K
                if not gated and rows < ops.PINGPONG_MIN_ROWS:
                    assert tile == 0, (rows, n, k)
            assert ops._pingpong_plan(16384, n, k, gated) == (256, 1), (n, k, gated)
    assert ops._pingpong_plan(2048, 4096, 4000 + 16, False) == (0, 1), "K must be whole stages of 32"
    assert ops._pingpong_plan(2048, 4096, 64, False) == (0, 1), "too few stages"
    assert ops._pingpong_plan(2048, 8192, 1024 + 32, False)[1] == 1, "a cut needs K % 64 == 0 and long ranges"


def test_plan_of_the_tiled_products():
    """The plan that the dispatch asks for: a tile that a kernel has (192 or 256 rows, or none), K cut only where every
    workgroup keeps a long range of whole stages and never for the gated product, few rows and shapes that the large tiles'
    kernel cannot take with the small tile, whose cuts are the small tile's own, tiles of 192 rows with K cut only where they
    leave fewer empty rows than 256, never for a near tie of the gated product, nor in one round over a short K where they
    have no empty rows to save; for the models' products and for odd sizes."""
    cus = ops.compute_units()
    shapes = [s for group in SHAPES.values() for s in group] + [(4096, 1024, False), (3072, 1024, True), (6144, 2560, False)]
    shapes += [(n, k, gated) for n in (8, 100, 131, 1000, 4100, 25000) for k in (32, 64, 96, 128, 160, 192, 1056, 4096, 8256, 17408)
               for gated in (False, True)]
    taken = set()
    for n, k, gated in shapes:
        for rows in (65, 90, 128, 129, 192, 193, 256, 257, 300, 385, 577, 700, 1000, 1025, 1318, 1536, 1800, 2049,
                     2096, 2850, 3333, 4614, 8192, 16384):
            tile, cut = ops._tiled_plan(rows, n, k, gated)
            where = (rows, n, k, gated, tile, cut)
            assert tile in (0, 192, 256), where
            assert not gated or cut == 1, where
            if tile == 0:
                assert cut == (ops._k_splits(rows, n, k, gated) if k % 64 == 0 else 1), where
                continue
            assert k % 32 == 0 and k >= 128 and cut in (1, 2, 4) and (gated or rows >= ops.PINGPONG_MIN_ROWS), where
            if cut > 1:
                assert k % 64 == 0 and (k // 32) % cut == 0 and k // cut >= ops.PINGPONG_SPLIT_MIN_K, where
            if tile == 192:
                assert k % 64 == 0 and (cut == 1 or -(-rows // 192) * 192 < -(-rows // 256) * 256), where
                t = lambda r: ops._large_us(rows, n, k, gated, r, 1)
                assert not gated or ops._pingpong_plan(rows, n, k, gated)[0] == 0 or t(192) < 0.98 * t(256), where
                tiles = -(-n // (128 if gated else 256)) * -(-rows // 192)
                if rows in (1318, 2096, 2850) and k < 4096 and cut == 1:  # just above whole tiles of 256, just below of 192
                    assert tiles > cus or ops._pingpong_plan(rows, n, k, gated)[0] == 0, where
            else:
                assert (tile, cut) == ops._pingpong_plan(rows, n, k, gated), where
            taken.add((tile, cut))
    assert {(192, 1), (192, 2), (192, 4), (256, 1), (256, 2), (256, 4)} <= taken, taken


def test_tiles_that_the_dispatch_asks_for():
    """Beside the plan's own: tiles the kernel has, wide last rows only for at most 128 of them, K in at most eight parts that
    all keep four stages or more, never for the gated product; few rows, K that is no multiple of 64 and a plan that
    was put in the place of the rule's own are left alone."""
    shapes = [s for group in SHAPES.values() for s in group] + [(100, 8256, False), (4100, 1056, False), (5120, 17408, False)]
    taken = set()
    for n, k, gated in shapes:
        for rows in (65, 256, 257, 280, 320, 385, 560, 631, 700, 900, 1100, 1320, 2100, 2600, 3111, 4614, 8192):
            plan = ops._tiled_plan(rows, n, k, gated)
            for normed in (False, True):
                tile, cut = ops._tiles(rows, n, k, gated, normed and not gated, *plan)
                where = (rows, n, k, gated, tile, cut)
                if (tile, cut) == plan:
                    continue
                assert rows >= ops.PINGPONG_MIN_ROWS and k % 64 == 0 and tile in (192, 256, ops.WIDE_LAST) and 1 <= cut <= ops.FINER_CUTS, where
                assert tile != ops.WIDE_LAST or 1 <= rows % 256 <= 128, where
                assert not gated or cut == 1, where
                stages = k // 32
                assert cut == 1 or (k // cut >= ops.PINGPONG_SPLIT_MIN_K and stages - -(-stages // cut) * (cut - 1) >= 4), where
                taken.add((tile, cut))
            other = (256, 2) if plan != (256, 2) else (192, 1)
            assert ops._tiles(rows, n, k, gated, False, *other) == other
    assert {t for t, _ in taken} == {192, 256, ops.WIDE_LAST} and {3, 5} <= {c for _, c in taken}, taken


def test_the_attention_plan_says_whether_the_runs_of_a_step_differ_much_in_keys():
    """One prompt from its start has runs of 128 to 2,048 keys (the portion kernel then cuts every run's keys over two
    groups of waves); a portion deep inside a long request, or several of them, has runs of about the same length."""
    from jllm_serve_amd.engine.step import Segment, StepBatch
    from jllm_serve_amd.parts.attention import GqaStepPlanner

    def facts(*portions):
        segments, row = [], 0
        for i, (n, pos0) in enumerate(portions):
            segments.append(Segment(f"r{i}", i, row, n, pos0, i))
            row += n
        batch = StepBatch(segments, row, len(segments), max(p + n for n, p in portions), 16, None, False)
        return GqaStepPlanner().plan(batch).facts

    assert facts((2048, 0))["key_groups"] == 2
    assert facts((1024, 0), (1024, 0))["key_groups"] == 2
    assert facts((2048, 6144))["key_groups"] == 1
    assert facts((2048, 2048))["key_groups"] == 1          # 2,176 to 4,096 keys: 1.3 times the average
    assert facts((512, 7680), (300, 0))["key_groups"] == 2  # a late portion beside a new prompt
    assert facts((1, 100), (1, 5000))["key_groups"] == 1   # single rows go to the split-key kernel anyway
    f = facts((2048, 0), (1, 77))
    assert f["key_groups"] == 2 and f["n_tiles_multi"] == 16 and f["single_rows"] == (2048, 1)


def test_attention_layers_of_several_head_counts_plan_once():
    """The runs of a step are cut and uploaded once whatever the layers' kv heads, under a key that any part can ask for by the
    planner's class; the counters are as many as the layer with the most kv heads takes."""
    from types import SimpleNamespace

    import torch
    from jllm_serve_amd.engine.step import ModelRunner, Segment, StepBatch
    from jllm_serve_amd.parts.attention import GqaStepPlanner
    planners = [GqaStepPlanner(n) for n in (2, 8, 4)]
    model = SimpleNamespace(step_planners=lambda: planners, device=torch.device("cpu"), config=SimpleNamespace(vocab=8))
    got = ModelRunner(model, None, 64).planners()
    assert [pl.key for pl in got] == [GqaStepPlanner.key]
    batch = StepBatch([Segment(i, i, i, 1, 9, i) for i in range(3)], 3, 3, 10, 16, None, False)
    assert len(got[0].plan(batch).arrays["arrivals"]) == 3 * 8


def test_plans_of_the_second_weight_streaming_kernel():
    """Every plan is one that the kernel has, parts of K are whole blocks that are all there, its counters fit the step's, and
    for up to 64 rows it knows nothing of their number; few columns and large products of many rows stay with the other kernels."""
    import inspect
    assert list(inspect.signature(ops._stream_plan.__wrapped__).parameters) == ["N", "K", "gated"]
    shapes = [s for v in SHAPES.values() for s in v] + [(4096, 1024, False), (3072, 1024, True), (1024, 3072, False), (2560, 9728, False), (16, 128, False),
                                                       (48, 1024, True), (151936, 4096, False)]
    taken = 0
    for n, k, gated in shapes:
        rows, parts = ops._stream_plan(n, k, gated)
        tiles = -(-n // (rows // 2 if gated else rows))
        assert rows in (32, 64, 96, 128) and 1 <= parts <= k // 128 and (parts == 1 or tiles <= ops.STREAM_COUNTERS), (n, k, gated, rows, parts)
        for m in (65, 100, 127, 128, 200, 333, 487, 640, 900, 1024, 1025, 4096):
            for adds in (False, True):
                plan = ops._wide_plan(m, n, k, gated, adds and not gated)
                if plan is None:
                    continue
                taken += 1
                rows, tile, parts = plan
                per = -(-(k // 128) // parts)
                assert rows in (32, 64, 96, 128) and tile in (64, 128) and m <= ops.WIDE_MOST_ROWS and k >= ops.WIDE_LEAST_K, (m, n, k, plan)
                assert -(-(k // 128) // per) == parts and (parts == 1 or -(-n // rows) * -(-m // tile) <= ops.STREAM_COUNTERS), (m, n, k, plan)
    assert taken > 20
    assert ops._wide_plan(487, 12288, 4096, True) is None and ops._wide_plan(300, 1024, 100, False) is None


def test_a_new_row_count_does_not_weigh_every_choice_again(monkeypatch):
    """The choices of the ring kernel for many rows cost the same for all row counts with the same tiles: the host weighs them once."""
    weighed = []
    estimate = ops._wide_us
    monkeypatch.setattr(ops, "_wide_us", lambda *args: weighed.append(args) or estimate(*args))
    for cached in (ops._wide_plan, getattr(ops, "_wide_best", ops._wide_plan)):
        cached.cache_clear()
    ops._wide_plan(449, 4096, 1024, False, 0)
    once = len(weighed)
    for m in range(450, 513):
        for adds in (0, 1, 2):
            ops._wide_plan(m, 4096, 1024, False, adds)
    assert 0 < once == len(weighed)


MANY = [s for v in SHAPES.values() for s in v] + [  # the smaller models' products, and odd sizes
    (4096, 1024, False), (1024, 2048, False), (3072, 1024, True), (1024, 3072, False), (6144, 2560, False), (2560, 9728, False), (3392, 2048, False),
    (12320, 2048, False), (22592, 4096, False), (8192, 2048, True)] + [(n, k, g) for n in (8, 131, 1000, 4100) for k in (32, 64, 96, 128, 192, 320, 1056, 4160, 8256)
                                                                      for g in (False, True)]


def test_choices_of_the_tiled_products():
    """What the dispatch asks for, at every row count of some and many of all shapes: a tile of a kernel that takes the sizes, K in no
    more parts than leave each one stages and never for the gated product, the norm's time counted where one is asked for; the same
    for all row counts of 32 with the same tiles, and the cheapest of the small kernel's choices by the estimate."""
    taken = set()
    for n, k, gated in MANY:
        rows_of = range(65, 1100, 7) if (n, k) in ((4096, 4096), (3392, 2048)) else (65, 96, 97, 128, 129, 192, 257, 288, 384, 385, 487, 513, 700, 1025, 1318, 1800, 2100, 3000, 8192)
        for rows in rows_of:
            for normed in (False,) if gated else (False, True):
                tile, cut, us = ops._own_choice(rows, n, k, gated, normed)
                where = (rows, n, k, gated, normed, tile, cut)
                taken.add((tile, cut))
                stages = -(-k // 64)
                assert cut == 1 or (not gated and stages > -(-stages // cut) * (cut - 1)), where
                if tile in (192, 256, ops.WIDE_LAST):
                    assert k % 32 == 0 and k >= 128 and k // cut >= 128, where
                    assert tile != ops.WIDE_LAST or (rows > 256 and 1 <= rows % 256 <= 128), where
                else:
                    assert tile in ops.SMALL_TILES and not (gated and tile == 64064), where
                assert ops._own_choice(-(-rows // 32) * 32, n, k, gated, normed)[:2] == (tile, cut), where
                if k % 64:
                    continue
                norm = ops._norm_us(rows, n) if normed and cut == 1 else 0.0
                assert abs(us - ops._tile_us(tile, rows, n, k, gated, cut) - norm) < 1e-6 * us, where
    assert len(taken) > 25 and {t for t, _ in taken} == {192, 256, ops.WIDE_LAST, *ops.SMALL_TILES}, taken


def test_what_the_large_tiles_decline_goes_to_the_best_small_one(monkeypatch):
    """An operand of 4 GB is none of the large tiles': the smaller ones take it in the tile and cut that are the cheapest of theirs, also with
    the norm of the new rows."""
    import torch

    import recorded
    seen = recorded.record(monkeypatch)
    monkeypatch.setattr(ops, "_try", lambda name, *args: seen.append((name, args)) or name != "jllm_gemm_pingpong_bf16")
    asked = 0
    for m, n, k in ((2048, 4096, 12288), (1800, 6144, 4096), (600, 5120, 17408), (8192, 4096, 4096)):
        a, w, res, gain = recorded.tensor(m, k), recorded.tensor(n, k), recorded.tensor(m, n, dtype=torch.float32), recorded.tensor(n)
        for normed, gated in ((False, False), (False, True), (True, False)):
            if ops._own_choice(m, n, k, gated, normed)[0] > 1000 or (normed and not ops._cut_takes_norm(m, n, k)):
                continue
            asked += 1
            small = ops._small_bests(-(-m // 64), n, k, gated)[normed][1:]
            del seen[:]
            if normed:
                with monkeypatch.context() as mp:
                    mp.setattr(torch.Tensor, "data_ptr", lambda self: 0)
                    ops.gemm_add_then_norm(a, w, res, gain, 1e-5, torch.bfloat16)
            else:
                ops.gemm(a, w, w2=w if gated else None, epilogue=ops.EPI_GATED if gated else ops.EPI_STORE)
            assert [name for name, _ in seen][0] == "jllm_gemm_pingpong_bf16", (m, n, k)
            if normed and small[1] == 1:
                continue  # K stays whole: the norm is a launch behind it
            name, args = seen[1]
            assert name == "jllm_gemm_mfma_bf16" and args[14:16] == small, (m, n, k, gated, normed, args[14:16], small)
    assert asked >= 6


def test_the_native_walks_find_the_cheapest():
    """The walks over the choices against every single one's time."""
    cus = ops.compute_units()
    for n, k, gated in MANY:
        if k % 64:
            continue
        for rows in (128, 320, 512, 832, 1216, 1344, 2112, 2560):
            for normed in (False, True):
                norm = lambda c: ops._norm_us(rows, n) if normed and c == 1 else 0.0
                all_ = []
                for tile in ops.SMALL_TILES:
                    r, c = divmod(tile, 1000)
                    groups = -(-n // (c // 2 if gated else c)) * -(-rows // r)
                    all_ += [(ops._tile_us(tile, rows, n, k, gated, cut) + norm(cut), tile, cut) for cut in ops.SMALL_CUTS if not (gated and tile == 64064)
                             and (cut == 1 or (not gated and k // cut >= ops.SMALL_CUT_MIN_K and groups * cut <= 3 * cus and k // 64 > -(-(k // 64) // cut) * (cut - 1)))]
                got = ops._small_bests(rows // 64, n, k, gated)[normed]
                assert got[1:] == min(all_)[1:] and abs(got[0] - min(all_)[0]) < 1e-9 * got[0], (rows, n, k, gated, normed)
                plan = ops._tiled_plan(rows, n, k, gated)
                if rows < ops.PINGPONG_MIN_ROWS or k < 128:
                    continue
                us = ops._tile_us(plan[0], rows, n, k, gated, plan[1]) + norm(plan[1]) if plan[0] else got[0]
                large = [(ops.FINER_AT_MOST * us, 0, 0)] + [
                    (ops._tile_us(tile, rows, n, k, gated, cut) + norm(cut), tile, cut) for tile in (192, 256, ops.WIDE_LAST) for cut in range(1, 2 if gated else ops.FINER_CUTS + 1)
                    if (cut == 1 or k // cut >= ops.PINGPONG_SPLIT_MIN_K) and not (tile == 192 and cut in (1, 2, 4)) and (tile != ops.WIDE_LAST or rows % 256 in (64, 128))]
                want = min(large)
                assert ops._finer_tiles(rows, n, k, gated, normed, *plan)[:2] == (want[1:] if want[1] else plan), (rows, n, k, gated, normed)
                assert ops._own_choice(rows, n, k, gated, normed)[2] < 1.05 * min(t for t, tile, _ in large if tile), (rows, n, k, gated, normed)


def test_a_prompt_of_a_new_length_costs_the_host_little(monkeypatch):
    """Of the tiled kernels' choices few are priced one by one in Python for a row count whose tiles were not seen, none for one whose
    tiles were."""
    priced = []
    estimate = ops._tile_us
    monkeypatch.setattr(ops, "_tile_us", lambda *args: priced.append(args) or estimate(*args))
    for cached in (f for f in vars(ops).values() if hasattr(f, "cache_clear") and f.__name__ in ("_own_choice", "_choice_of", "_small_bests", "_wide_plan", "_wide_best")):
        cached.cache_clear()
    for n, k, gated in ((4096, 1024, False), (1024, 2048, False), (3072, 1024, True), (4096, 4096, False), (4096, 12288, False)):
        for rows in (487, 833, 1500):
            ask = lambda m: [ops._cut_takes_norm(m, n, k) if not gated else None, ops._wide_plan(m, n, k, gated, 0), ops._tiled_choice(m, n, k, gated, False)]
            del priced[:]
            ask(rows)
            assert len(priced) <= 16, (n, k, gated, rows, len(priced))
            del priced[:]
            for m in range(-(-rows // 32) * 32 - 31, -(-rows // 32) * 32 + 1):
                ask(m)
            assert not priced, (n, k, gated, rows)


def test_ranges_of_the_latent_attention_of_single_rows():
    """Whole blocks of 64 keys, no more ranges than the merge takes and enough for the span wherever it lies, about two workgroups a compute
    unit at most; ranges of one block only where rows as long as they may be have one compute unit each."""
    cus = ops.compute_units()
    for rows in (1, 2, 3, 5, 8, 11, 15, 16, 17, 24, 31, 32, 48, 64, 100, 128, 200, 255, 256, 257, 600):
        for heads in (1, 5, 16, 32, 64, 65, 128, 200):
            for window in (0, 100, 256, 300, 1000, 1024, 4096, 50000):
                for longest in (16, 255, 256, 257, 512, 768, 1024, 2048, 8192, 16000, 131072, 1 << 20):
                    split, n_z = ops._latent_split(rows, heads, window, longest)
                    where = (rows, heads, window, longest, split, n_z)
                    windowed = 0 < window < longest
                    span = window if windowed else longest
                    groups = rows * -(-heads // 64)
                    if split == 0:
                        assert n_z == 1 and (span < ops.LATENT_SPAN_MIN or span <= 256 or groups >= cus), where
                        continue
                    assert split % 64 == 0 and 2 < n_z <= 64 and (n_z - 1) * split >= span, where
                    assert split > 64 or groups * (n_z - 1 + windowed) <= cus, where
                    assert groups * (n_z - 1) < 2 * cus + groups, where


def test_order_of_the_tiles_of_odd_numbers_of_columns():
    """Every tile is taken once, whatever the numbers; with an odd number of columns, and with two more than a multiple of four, the
    workgroups of a die (every eighth) share the weights of as few columns as their number allows."""
    import ctypes
    place = ops.library().jllm_tiled_place
    out = (ctypes.c_int * 2)()
    for rows, cols in ((1, 1), (1, 53), (2, 3), (5, 53), (7, 53), (7, 27), (18, 27), (3, 97), (9, 25), (8, 89), (13, 10), (4, 20), (5, 16), (40, 9), (300, 7), (70, 177)):
        taken, dies = set(), [set() for _ in range(8)]
        for b in range(rows * cols):
            assert place(rows, cols, b, out) == 0
            taken.add((out[0], out[1]))
            dies[b % 8].add(out[1])
        assert taken == {(r, c) for r in range(rows) for c in range(cols)}, (rows, cols)
        if rows > 1 and cols % 4:
            most = -(-rows * cols // 8)
            assert max(map(len, dies)) <= (most + rows - 2) // rows + 1, (rows, cols)
    assert place(4, 20, 80, out) == -1


def test_declared_arguments_are_those_of_the_sources():
    """Every entry point's declared argument types against its definition: a pointer declared as an int would reach the
    kernel cut to 32 bits."""
    import ctypes
    import os
    import re
    from jllm_serve_amd.kernels import build
    kinds = {ctypes.c_void_p: "pointer", ctypes.c_int: "int", ctypes.c_float: "float", ctypes.c_longlong: "long", ctypes.c_long: "long"}
    defined = {}
    for name in build.sources():
        with open(os.path.join(build.SRC_DIR, name)) as f:
            for fn, args in re.findall(r'extern "C" int (\w+)\(([^)]*)\)\s*{', f.read()):
                defined[fn] = ["pointer" if "*" in a or "hipStream_t" in a else "float" if "float" in a else
                               "long" if re.search(r"\b(long|size_t|int64_t)\b", a) else "int" for a in args.split(",") if a.strip()]
    declared = {**ops._SIGS, **ops._OPTIONAL_SIGS}
    assert len(declared) > 40 and set(declared) <= set(defined), set(declared) - set(defined)
    for fn, args in declared.items():
        assert [kinds[a] for a in args] == defined[fn], fn
