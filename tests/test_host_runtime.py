"""What the host side does around the kernels, looked at without a GPU: a stand-in for the HIP runtime (host_hip.py) logs
the launches, allocations and graphs."""
import pytest

import host_hip


@pytest.mark.parametrize("captured", [True, False], ids=["captured", "eager"])
def test_passes_of_two_threads_do_not_interleave(captured):
    """Every pass writes the same arena, so the launches of one run_async may not stand between those of another."""
    host_hip.run('''
    import threading
    mdl = model.Model(model.Graph.from_spec(zoo.config2_mbv2_block()), 2)
    mdl.run()
    if %d:
        assert mdl.enable_graph()
    hip.host_hip_clear()
    mdl.run_async()
    one = [l["name"] for l in launches()]
    assert len(one) > 1
    hip.host_hip_clear()
    hip.host_hip_delay(200)
    start = threading.Barrier(2)

    def passes():
        start.wait()
        for _ in range(40):
            mdl.run_async()

    threads = [threading.Thread(target=passes) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    log = launches()
    assert len(log) == 80 * len(one) and len({l["thread"] for l in log}) == 2
    for i in range(0, len(log), len(one)):
        part = log[i:i + len(one)]
        assert [l["name"] for l in part] == one and len({l["thread"] for l in part}) == 1, i
    ''' % captured)


def test_a_plan_replayed_as_launches_makes_no_graph_exec():
    """enable_graph instantiates only what run_async launches: a short plan is replayed from its launch list, a plan of
    many small launches as the graph."""
    host_hip.run('''
    def enabled(spec, batch):
        mdl = model.Model(model.Graph.from_spec(spec), batch)
        hip.host_hip_clear()
        assert mdl.enable_graph() and mdl.enable_graph()  # (the second call finds it done)
        made = hip.host_hip_calls(b"hipGraphInstantiate")
        hip.host_hip_clear()
        mdl.run()
        replayed = hip.host_hip_launches(), hip.host_hip_calls(b"hipGraphLaunch")
        mdl.disable_graph()
        hip.host_hip_clear()
        mdl.run()
        return made, replayed, hip.host_hip_launches()

    made, (plain, graphs), eager = enabled(zoo.config1_single_conv(), 1)
    assert (made, plain, graphs, eager) == (0, 1, 0, 1)
    made, (plain, graphs), eager = enabled(zoo.config3_mobilenetv2(resolution=96), 1)
    assert (made, plain, graphs) == (1, 0, 1) and eager > 24
    ''')


def test_memory_queries_count_the_workspace_and_the_staging():
    """A block run as two launches keeps its depthwise result in the model's workspace, and host copies pass through
    pinned memory of the model's own: both are the model's memory."""
    out = host_hip.run('''
    spec = zoo.config2_mbv2_block()
    mdl = model.Model(model.Graph.from_spec(spec), 2)
    before = mdl.device_bytes()
    mdl.run()
    assert len(launches()) == 2
    assert mdl.device_bytes() == before + 2 * 56 * 56 * 144, (before, mdl.device_bytes())
    m.model.lib().espdl_model_print_profile(mdl.h)  # nothing was copied yet
    mdl.get_tensor(spec.outputs[0])                 # too large for the staging
    m.model.lib().espdl_model_print_profile(mdl.h)
    spec = zoo.config3_mobilenetv2(resolution=96)
    small = model.Model(model.Graph.from_spec(spec), 1)
    small.get_tensor(spec.outputs[0])
    m.model.lib().espdl_model_print_profile(small.h)
    ''')
    pinned = [int(line.split()[2]) for line in out.splitlines() if line.startswith("host memory:")]
    assert pinned == [0, 0, 65536]


@pytest.mark.parametrize("round_mode", [0, 1], ids=["half_up", "half_even"])
def test_fused_blocks_with_clips_have_a_kernel(round_mode):
    """What fuse_dw_project joins must have a launch in the model's rounding mode: pointwise blocks with and without a single
    launch, and a stem in front of the first block (the kernels are not run here)."""
    host_hip.run("""
    import test_gpu_model
    for shape, exp, out, stride, stem, batch in [((56, 56, 24), 144, 24, 1, False, 2), ((56, 56, 24), 144, 24, 1, False, 256),
                                                 ((28, 28, 32), 192, 64, 2, False, 4), ((14, 14, 64), 384, 64, 1, False, 3),
                                                 ((224, 224, 3), 32, 16, 1, True, 2)]:
        spec = test_gpu_model.clip_block(shape, exp, out, stride, stem)
        mdl = model.Model(model.Graph.from_spec(spec), batch, round_mode=%d)
        mdl.run()  # raises where a module's launch is refused
        mdl.close()
    """ % round_mode)


def test_wide_filter_walks_ask_for_lds_that_the_kernel_may_have():
    """A launch past 64 KB of LDS (34848 bytes of the kernel's own and the walk's constants) needs the kernel's limit raised;
    walks of 9 to 12 steps."""
    host_hip.run("""
    for rows, filters, steps in [(20480, 6625, 9), (20003, 2305, 10), (20480, 2563, 11), (30000, 2817, 12)]:
        desc = m.capi.make_desc((rows, 1, 1, 64), filters, (1, 1))
        hip.host_hip_clear()
        rc = m.lib().espdl_hip_conv2d(ctypes.byref(desc), 1 << 20, 1 << 30, None, 1 << 31, None, 1 << 32, None)
        log = launches()
        assert rc == 0 and len(log) == 1 and "conv2d_s8_wide" in log[0]["name"], (rc, log)
        assert log[0]["lds"] == 3 * 4 * 256 * steps
        assert 34848 + log[0]["lds"] <= 65536 or log[0]["limit"] >= log[0]["lds"], log
    """)


def test_wide_filters_walk_several_times_where_the_shares_stay_even():
    """The layers that take longer with several walks to a workgroup keep a workgroup per walk (us: several, one): one compute
    unit would get more tiles than before, or the last filters leave too many of them idle."""
    host_hip.run("""
    for rows, channels, filters, several in [(20480, 120, 6625, True),   # 42.4, 46.6
                                             (20480, 128, 6625, True),   # 52.6, 55.5
                                             (20493, 120, 6625, True), (20493, 64, 6625, True), (33000, 64, 4509, True),
                                             (11520, 72, 6625, False),   # 34.7, 31.7
                                             (17602, 91, 3327, False),   # 43.5, 40.5
                                             (10944, 125, 6909, False),  # 86.1, 79.5
                                             (1024, 48, 6625, False)]:   # one round
        desc = m.capi.make_desc((rows, 1, 1, channels), filters, (1, 1))
        hip.host_hip_clear()
        rc = m.lib().espdl_hip_conv2d(ctypes.byref(desc), 1 << 20, 1 << 30, None, 1 << 31, None, 1 << 32, None)
        log = launches()
        build = "conv2d_s8_wide_kernelILi%dELb%dE" % (1 if channels <= 64 else 2, several)
        assert rc == 0 and len(log) == 1 and build in log[0]["name"], (rows, channels, log)
        assert (log[0]["grid"][0] < (rows + 63) // 64) == several, (rows, channels, log)
    """)


def test_depthwise_strips_are_found_quickly():
    """The strip count of the depthwise row walks is the cheapest of all (the plain search below), and finding it does not
    take longer than the launch: a layer of a million rows."""
    host_hip.run('''
    import math, time

    def launch(n, h, w, c, stride=1):
        desc = m.capi.make_desc((n, h, w, c), c, (3, 3), (stride, stride), pads=(1, 1, 1, 1), group=c)
        hip.host_hip_clear()
        t = time.perf_counter()
        rc = m.lib().espdl_hip_conv2d(ctypes.byref(desc), 1 << 20, 1 << 40, None, 1 << 41, None, 1 << 42, None)
        t = time.perf_counter() - t
        log = launches()
        assert rc == 0 and len(log) == 1 and "strip" in log[0]["name"], (rc, log)
        return log[0]["grid"][0], t

    for n, h, w, c, stride in [(1, 1, 1, 4, 1), (1, 7, 7, 960, 1), (37, 14, 14, 384, 1), (256, 56, 56, 144, 1), (256, 112, 112, 96, 2),
                               (3, 97, 55, 61, 2), (512, 20, 80, 24, 1), (1, 4096, 1, 20, 1), (2, 3001, 7, 5, 1), (1, 1009, 3, 4, 2)]:
        out_h, out_w = (h - 1) // stride + 1, (w - 1) // stride + 1
        per_strip, best = n * ((out_w + 3) // 4) * ((c + 3) // 4), None
        for s in range(1, out_h + 1):
            rows = -(-out_h // s)
            cost = math.ceil(per_strip * s / (64 * 4 * 4 * 256)) * (rows + 2.5)
            if -(-out_h // rows) == s and (best is None or cost < best[0]):
                best = cost, s
        blocks = -(-per_strip * best[1] // 256)
        if n * h * w * c >= 64 << 20:
            blocks = 8 * -(-blocks // 8)
        assert launch(n, h, w, c, stride)[0] == blocks, (n, h, w, c, stride)
    fastest = min(launch(1, 1 << 20, 1, 4)[1] for _ in range(5))
    assert fastest < 1e-3, fastest
    ''')


def test_pool_strips_are_found_quickly():
    """The same for the strips of the stride-1 max pool."""
    host_hip.run('''
    import math, time

    def launch(n, h, w, c, k):
        hip.host_hip_clear()
        t = time.perf_counter()
        rc = m.lib().espdl_hip_max_pool_pitched(1 << 20, 8, n, h, w, c, k, k, 1, 1, k // 2, (k - 1) // 2, k // 2, (k - 1) // 2, 0, 0, 1 << 42, None)
        t = time.perf_counter() - t
        log = launches()
        assert rc == 0 and len(log) == 1 and "max_pool_s8_window" in log[0]["name"], (rc, log)
        return log[0]["grid"][0] * log[0]["block"][0], t

    for n, h, w, c, k in [(1, 1, 1, 8, 3), (64, 20, 20, 128, 5), (327, 80, 80, 128, 5), (256, 56, 56, 144, 5), (128, 36, 8, 194, 5),
                          (2, 3001, 7, 24, 3), (1, 4096, 1, 16, 2), (5, 97, 31, 9, 2)]:
        vec = 16 if c >= 16 and c != 24 else 8
        per_row, best, score = n * ((w + 1) // 2) * -(-c // vec), 1, -1.0
        for s in range(1, h + 1):
            rows = -(-h // s)
            if -(-h // rows) != s:
                continue
            rounds = per_row * s / 64.0 / (256 * 4 * 4)
            here = rounds / int(rounds + 0.999999) / (1.0 + 0.5 * (k - 1) / rows)
            if here > score * 1.02:
                score, best = here, s
        assert launch(n, h, w, c, k)[0] == -(-per_row * best // 256) * 256, (n, h, w, c, k)
    fastest = min(launch(1, 1 << 20, 1, 64, 5)[1] for _ in range(5))
    assert fastest < 1e-3, fastest
    ''')


def test_pools_of_one_row_keep_neighbouring_wavefronts_together():
    """Strips of one row: single wavefronts only while the device has two of them per compute unit (us with single wavefronts
    and with four to a workgroup)."""
    host_hip.run('''
    for n, h, w, c, k, threads in [(1, 13, 13, 128, 5, 64),   # 2.9, 3.2
                                   (1, 30, 30, 198, 5, 64),
                                   (12, 96, 54, 32, 3, 256),  # 4.67, 3.6
                                   (7, 72, 24, 128, 3, 256),  # 4.40, 3.5
                                   (87, 12, 18, 80, 3, 256)]:
        hip.host_hip_clear()
        rc = m.lib().espdl_hip_max_pool_pitched(1 << 20, 8, n, h, w, c, k, k, 1, 1, k // 2, (k - 1) // 2, k // 2, (k - 1) // 2, 0, 0, 1 << 42, None)
        log = launches()
        assert rc == 0 and len(log) == 1 and "max_pool_s8_window_row" in log[0]["name"], (rc, log)
        assert log[0]["block"][0] == threads and log[0]["grid"][0] * threads <= (32768 if threads == 64 else 1 << 30), (n, h, w, c, k, log)
    ''')


def test_narrow_kernels_stay_inside_the_grid_limit():
    """A launch has fewer than 2^32 threads along x: layers with more pixels than that go to the kernel with larger tiles."""
    host_hip.run('''
    for dtype in (8, 16):
        for n, h, w, c, oc, k in [(1500, 1000, 1000, 1, 8, (5, 1)), (700, 1000, 1000, 1, 8, (5, 1)), (1, 9, 9, 1, 8, (5, 1))]:
            if dtype == 16 and n > 700:
                continue
            desc = m.capi.make_desc((n, h, w, c), oc, k, pads=(2, 2, 0, 0), dtype=dtype)
            hip.host_hip_clear()
            rc = m.lib().espdl_hip_conv2d(ctypes.byref(desc), 1 << 36, 1 << 37, None, 1 << 38, None, 1 << 39, None)
            log = launches()
            assert rc == 0 and log, (rc, n)
            for l in log:
                assert l["grid"][0] * l["block"][0] < 1 << 32, (dtype, n, l)
    ''')


@pytest.mark.parametrize("spec,batch", [("config4_yolo_style(resolution=96)", 1), ("config1_single_conv()", 1),
                                        ("config2_mbv2_block()", 2)], ids=["shared launches", "one convolution", "block"])
def test_a_pass_in_an_open_group_of_convolutions_fails(spec, batch):
    """The group would hold back the pass's convolutions while the modules that read them run: every way to run the plan fails
    and launches nothing, and works again behind the group."""
    host_hip.run('''
    L, spec = m.lib(), zoo.%s
    mdl = model.Model(model.Graph.from_spec(spec), %d)

    def passes():
        ways = {"run": mdl.run, "run_async": mdl.run_async, "enable_graph": mdl.enable_graph, "profile": lambda: mdl.profile(1)}
        for name, way in ways.items():
            hip.host_hip_clear()
            try:
                done = way()
                done = len(done) > 0 if name == "profile" else done in (None, True)
            except model.EspdlModelError:
                done = False
            yield name, done, hip.host_hip_launches(), hip.host_hip_calls(b"hipGraphLaunch")
            if name == "enable_graph":
                mdl.disable_graph()

    def replay():
        hip.host_hip_clear()
        try:
            mdl.run()
        except model.EspdlModelError:
            return False, hip.host_hip_launches(), hip.host_hip_calls(b"hipGraphLaunch")
        return True, hip.host_hip_launches(), hip.host_hip_calls(b"hipGraphLaunch")

    mdl.run()
    assert L.espdl_hip_conv2d_group_begin() == 0
    for name, done, n, graphs in passes():
        assert not done and n == 0 and graphs == 0, (name, done, n)
    hip.host_hip_clear()
    assert L.espdl_hip_conv2d_group_end() == 0 and hip.host_hip_launches() == 0  # nothing was held back either
    for name, done, n, graphs in passes():
        assert done and n + graphs > 0, (name, done, n)
    assert mdl.enable_graph() and replay()[0]
    assert L.espdl_hip_conv2d_group_begin() == 0
    assert replay() == (False, 0, 0)
    assert L.espdl_hip_conv2d_group_end() == 0
    assert replay()[0]
    ''' % (spec, batch))


def test_other_calls_refuse_in_an_open_group():
    """What a group holds back may be read by any other launch: every call of the header that takes a stream, but the three
    that a group is made of, fails before it looks at its arguments."""
    host_hip.run('''
    import re
    text = re.sub(r"/\\*.*?\\*/", "", open(sys.path[0] + "/include/espdl_hip.h").read(), flags=re.S)
    calls = {name: args.count(",") + 1 for name, args in re.findall(r"\\bint (espdl_hip_\\w+)\\(([^)]*)\\)", text) if "void *stream" in args}
    members = {"espdl_hip_conv2d", "espdl_hip_conv2d_add", "espdl_hip_conv2d_s16_x8"}
    assert len(calls) > 40 and members < set(calls)
    L = m.lib()
    message = L.espdl_hip_last_error
    assert L.espdl_hip_conv2d_group_begin() == 0
    for name, n in calls.items():
        call = getattr(ctypes.CDLL(m.capi.LIB_PATH), name)  # (a handle without argument types)
        assert call(*[ctypes.c_void_p(0)] * n) == -22, name
        assert (name.encode() + b" in an open group" in message()) == (name not in members), (name, message())
    assert hip.host_hip_launches() == 0
    assert L.espdl_hip_conv2d_group_end() == 0
    for name, n in calls.items():
        getattr(ctypes.CDLL(m.capi.LIB_PATH), name)(*[ctypes.c_void_p(0)] * n)
        assert b"in an open group" not in message(), (name, message())
    ''')


def test_a_block_in_an_open_group_is_refused():
    """Its project layer is a narrow convolution: the group would keep it."""
    host_hip.run('''
    d = m.capi.MbconvDesc(1, 14, 14, 64, 384, 64, 1, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 0, 0, 1, 1, 1)
    base = 1 << 30
    w = m.capi.MbconvWeights(base * 3, None, base * 4, base * 5, None, base * 6, base * 7, None, base * 8)
    call = lambda: m.lib().espdl_hip_mbconv_s8_ws(ctypes.byref(d), base, ctypes.byref(w), None, base * 2, base * 10, None)
    assert m.lib().espdl_hip_mbconv_s8_workspace(ctypes.byref(d)) > 0
    assert call() == 0 and len(launches()) == 2
    hip.host_hip_clear()
    assert m.lib().espdl_hip_conv2d_group_begin() == 0
    assert call() == -22 and len(launches()) == 0
    assert m.lib().espdl_hip_conv2d_group_end() == 0 and len(launches()) == 0
    ''')


def test_two_launch_cases_take_the_tile_of_their_name():
    """The builds of the expand + depthwise launch that test_gpu_kernels.py means to run."""
    host_hip.run('''
    import re
    import test_gpu_kernels
    taken = set()
    for name, (n, h, w, cin), ce, cout, stride, res, half_even, extra in test_gpu_kernels.TWO_LAUNCH_TILES:
        d = m.capi.MbconvDesc(n, h, w, cin, ce, cout, 1, 3, 3, stride, stride, 1, 1, 1, 1, 1, 1, 1, 1, 0, int(half_even), ce, ce, cout)
        if extra == "clip":
            d.clip_expand = d.clip_dw = 1
            d.clip_expand_max = d.clip_dw_max = 90
        base = 1 << 30
        weights = m.capi.MbconvWeights(base * 3, None, base * 4, base * 5, None, base * 6, base * 7, None, base * 8)
        hip.host_hip_clear()
        assert m.lib().espdl_hip_mbconv_s8_ws(ctypes.byref(d), base, ctypes.byref(weights), base * 9 if res else None, base * 2, base * 10, None) == 0
        build = re.search("kernelILi(.*?)ELi(.*?)ELi(.*?)ELi(.*?)ELb(.)ELb(.)ELb(.)E", launches()[0]["name"]).groups()
        rows, columns = re.match("([0-9]+)_rows_([0-9]+)", name).groups()
        want = rows, columns, "2" if "_s2" in name else "1", str(-(-cin // 64)), str(int(half_even)), str(int(extra == "clip")), str(int("loop" in name))
        assert build == want, (name, build)
        taken.add((build[0], build[1], build[2], build[6]))
    assert len(taken) == 12, taken  # nine tiles, three of them with the loop too
    ''')


def test_layers_that_share_a_launch():
    """What a pass of small graphs launches: the early layer goes out with the first one, and a pass module by module with its own
    place's neighbours."""
    host_hip.run('''
    import test_gpu_model
    expected = {"in_place": 4, "slices": 4, "residual": 3, "unread": 4}
    for kind, launched in expected.items():
        mdl = model.Model(model.Graph.from_spec(test_gpu_model.shared_launch_graph(kind)), 2)
        hip.host_hip_clear()
        mdl.run()
        names = [l["name"] for l in launches()]
        assert len(names) == launched and sum("narrow_group" in n for n in names) == 1, (kind, names)
        assert "narrow_group" in names[1], (kind, names)  # behind the trunk
        hip.host_hip_clear()
        mdl.profile(1)  # four passes of it
        names = [l["name"] for l in launches()]
        assert not any("narrow_group" in n for n in names) and len(names) == 4 * (launched + 1), (kind, names)
        mdl.close()
    ''')


def test_layers_run_early_only_while_the_arena_stays_small():
    """A layer that runs in front of its place keeps its output until there: up to a sixteenth of the arena and 4 MB."""
    host_hip.run('''
    import test_gpu_model
    output = 4 * 20 * 20 * 64  # of a side layer

    def plan(side):
        spec = test_gpu_model.shared_launch_graph("side", side)
        mdl = model.Model(model.Graph.from_spec(spec), 4)
        parameters = sum(data.nbytes for _, _, data, _ in spec.initializers.values())
        hip.host_hip_clear()
        mdl.run()
        shared = any("narrow_group" in l["name"] for l in launches())
        arena = mdl.device_bytes() - parameters
        mdl.close()
        return shared, arena

    shared, few = plan(30)
    assert shared and few > 20 * output
    shared, many = plan(90)
    assert not shared and many < 20 * output, many
    ''')


def test_residual_walks_take_four_filter_tiles_only_where_they_gain():
    """Filter tiles of the walking kernel's build for 3 x 3 layers with a residual operand (in microseconds: two tiles, four)."""
    host_hip.run('''
    for shape, oc, tiles in [((58, 40, 40, 64), 128, 2),   # 14.2, 17.4
                             ((110, 40, 40, 40), 64, 2),   # 13.5, 16.3
                             ((64, 80, 80, 64), 64, 4),    # 38, 30
                             ((216, 104, 104, 48), 64, 4),
                             ((244, 41, 37, 64), 64, 4), ((130, 37, 45, 52), 128, 4), ((256, 39, 43, 44), 64, 4)]:
        pads = {45: (0, 1, 0, 1), 43: (2, 0, 2, 1)}.get(shape[2], (1, 1, 1, 1))
        desc = m.capi.make_desc(shape, oc, (3, 3), pads=pads, n_shift=oc)
        for pitches in ((0, 0, 0), (192, 192, 192)):  # slices of wider tensors
            if pitches[0] and shape[1:] != (80, 80, 64):
                continue
            desc.in_pitch, desc.out_pitch, desc.res_pitch = pitches
            hip.host_hip_clear()
            rc = m.lib().espdl_hip_conv2d_add(ctypes.byref(desc), 1 << 36, 1 << 37, None, 1 << 38, None, 1 << 39, 1 << 40, None)
            names = [l["name"] for l in launches()]
            assert rc == 0 and len(names) == 1, (shape, names)
            assert "conv2d_s8_walk_kernelILi3ELi1ELi%dELi%dELb1E" % ((shape[3] + 15) // 16, tiles) in names[0], (shape, pitches, names)
    ''')


def test_windows_over_channels_that_are_no_multiple_of_four_go_to_the_faster_kernel():
    """The kernel of a few pixels against the tiled GEMM and the first-layer kernel (their microseconds beside the layer)."""
    host_hip.run('''
    L = m.lib()
    L.espdl_hip_conv2d_s8_kernel.restype = ctypes.c_char_p
    at = ctypes.c_void_p(256)
    for shape, oc, k, stride, residual, kernel in [((19, 14, 14, 87), 444, 5, 2, None, b"unitgemm"),   # 41, 20
                                                   ((16, 20, 20, 258), 64, 3, 1, None, b"unitgemm"),   # 32, 21
                                                   ((4, 40, 40, 94), 64, 5, 1, at, b"unitgemm"),       # 29, 21
                                                   ((10, 26, 26, 33), 64, 3, 1, at, b"unitgemm"),      # 8.9, 6.8
                                                   ((7, 52, 52, 221), 35, 1, 2, at, b"narrow"),        # 6.2, 6.5
                                                   ((205, 4, 41, 7), 6, 3, 1, None, b"narrow"),        # 5.7, 7.2
                                                   ((91, 40, 40, 13), 14, 3, 1, None, b"narrow"),      # 12.2, 15.4
                                                   ((7, 47, 86, 5), 7, 3, 1, None, b"narrow"),         # 4.8, the first-layer kernel 7.7
                                                   ((6, 104, 104, 4), 41, 3, 2, None, b"narrow"),      # 4.8, 11.3
                                                   ((19, 52, 52, 2), 8, 3, 1, None, b"stem"),          # 5.7, 5.7
                                                   ((1, 13, 13, 33), 64, 3, 1, None, b"narrow")]:
        desc = m.capi.make_desc(shape, oc, (k, k), (stride, stride), pads=(k // 2,) * 4, n_shift=oc)
        name = L.espdl_hip_conv2d_s8_kernel(ctypes.byref(desc), at, at, None, residual, at)
        assert name == b"conv2d_s8_" + kernel, (shape, name)
    ''')
