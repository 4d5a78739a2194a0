"""The flat step (pamhd_set_launch bit 7 and the default of small grids: one
launch for all faces, one for all cells) against the FP64 oracle, and in
mixed precision against the accumulating marches, bit for bit: row lengths
around the block of 256 threads and the wave of 64, grids of one cell,
steps that alternate with the other step structures (which carry the lagged
speeds in another form), and the first failing face in index order."""
import numpy as np
import pytest

import oracle_lib as O

SOLVERS = [("rusanov", O.RUSANOV), ("hll-athena", O.HLL), ("hlld-athena", O.HLLD),
           ("roe-athena", O.ROE)]
SHAPES = [(1, 1, 1), (5, 3, 4), (63, 2, 2), (64, 4, 1), (257, 1, 1), (17, 15, 1), (1, 1, 300),
          (65, 30, 1), (64, 32, 64), (67, 31, 64)]


def _state(cells, seed=5):
    from pamhd_amd import configs
    return configs.orszag_tang_vortex(cells, noise=0.02, seed=seed)


@pytest.mark.parametrize("d", [1, 2, 3, 5, 7, 25, 64, 127, 256, 641, 65535, (1 << 27) + 1, (1 << 28) - 1])
def test_flat_index_division_is_exact(d):
    """q = (c * m) >> sh with sh = 28 + ceil(log2 d), m = floor(2^sh / d) + 1
    (FlatDiv) at the ends of every quotient's range that 28-bit indexes reach"""
    sh = 28 + max(0, (d - 1).bit_length())
    m = ((1 << sh) // d) + 1
    assert m < 1 << 32
    top = (1 << 28) - 1
    q = np.unique(np.linspace(0, top // d, 4001).astype(np.int64))
    for c in (q * d, q * d + d - 1):
        c = c[c <= top]
        assert all((int(x) * m) >> sh == int(x) // d for x in c)


@pytest.mark.gpu
@pytest.mark.parametrize("cells", SHAPES)
@pytest.mark.parametrize("name,sid", SOLVERS)
def test_flat_fp64_bit_exact_vs_oracle(gpu, cells, name, sid):
    from pamhd_amd import solver as S
    state, length, gamma, mu0 = _state(cells)
    n = state.shape[1]
    bg = 0.1 * np.random.default_rng(3).normal(size=(9, n)) if name in ("rusanov", "hll-athena") else None
    ref = state.copy()
    og = O.make_grid(cells, length, gamma, mu0, bg)
    st, steps, t = O.run_periodic(og, sid, 0.3, 0.0, 1e9, ref, max_steps=4)
    assert st == 0
    with S.Grid(cells, length, gamma, mu0) as g:
        g.set_launch(128)
        if bg is not None:
            g.set_background_faces(bg)
        g.upload(state)
        print("cells", cells, name, flush=True)
        assert g.run(name, 0.3, 0.0, 1e9, max_steps=4) == (steps, t)
        np.testing.assert_array_equal(g.download(), ref)
        assert g.last_flux_calcs() == 3 * n


@pytest.mark.gpu
@pytest.mark.parametrize("cells", [(128, 128, 56), (128, 128, 57), (130, 128, 57)])
@pytest.mark.parametrize("name", ["rusanov", "hll-athena"])
def test_background_steps_match_the_flat_step(gpu, cells, name):
    """the default step with a background field around 7 2^17 cells, where
    grids of full tiles leave the flat step, against the flat step"""
    from pamhd_amd import solver as S
    state, length, gamma, mu0 = _state(cells)
    bg = 0.1 * np.random.default_rng(3).normal(size=(9, state.shape[1]))
    out = []
    for flat in (True, False):
        with S.Grid(cells, length, gamma, mu0) as g:
            if flat:
                g.set_launch(128)
            g.set_background_faces(bg)
            g.upload(state)
            print("cells", cells, name, "flat", flat, flush=True)
            out.append((g.run(name, 0.3, 0.0, 1e9, max_steps=3), g.max_signal_speeds(), g.download()))
    assert out[0][:2] == out[1][:2]
    np.testing.assert_array_equal(out[0][2], out[1][2])


@pytest.mark.gpu
@pytest.mark.parametrize("cells", [(64, 12, 10), (70, 13, 3), (33, 21, 20)])
@pytest.mark.parametrize("name", [s[0] for s in SOLVERS])
def test_flat_mixed_matches_marches(gpu, cells, name):
    """(the other solvers' passes, with a background field where there is one)"""
    from pamhd_amd import solver as S
    state, length, gamma, mu0 = _state(cells)
    bg = 0.1 * np.random.default_rng(3).normal(size=(9, state.shape[1])) if name in ("rusanov", "hll-athena") else None
    out = []
    for flat in (True, False):
        with S.Grid(cells, length, gamma, mu0, precision="mixed") as g:
            g.set_launch(128) if flat else g.set_fused_step("accumulate")
            if bg is not None:
                g.set_background_faces(bg)
            g.upload(state)
            print("cells", cells, name, "flat", flat, flush=True)
            out.append((g.run(name, 0.3, 0.0, 1e9, max_steps=6), g.max_signal_speeds(),
                        g.download()))
    assert out[0][:2] == out[1][:2]
    np.testing.assert_array_equal(out[0][2], out[1][2])


@pytest.mark.gpu
def test_flat_steps_between_other_steps(gpu):
    """lagged step lengths carry over from flat steps to the others, fixed
    steps and an autotuning run, and back"""
    from pamhd_amd import solver as S
    cells = (40, 9, 17)
    state, length, gamma, mu0 = _state(cells)

    def go(flat):
        with S.Grid(cells, length, gamma, mu0) as g:
            g.upload(state)
            dts = []
            for k in range(9):
                if flat and k % 3 == 1:
                    g.set_fused_step("passes" if k == 4 else "accumulate")
                elif flat:
                    g.set_launch(128)
                else:
                    g.set_fused_step("passes")
                if k == 6:
                    g.step_fixed("hlld-athena", 1e-4)
                if k == 7 and flat:
                    g.autotune("hlld-athena")
                dts.append(g.step("hlld-athena", 0.0 if k == 0 else 1e300, 0.3))
            return dts, g.max_signal_speeds(), g.download()

    a, b = go(True), go(False)
    assert a[0] == b[0] and a[1] == b[1] and a[0][1] > 0
    np.testing.assert_array_equal(a[2], b[2])


@pytest.mark.gpu
def test_flat_reports_the_first_failing_face(gpu):
    from pamhd_amd import _lib
    from pamhd_amd import solver as S
    cells = (64, 12, 10)
    state, length, gamma, mu0 = _state(cells, 9)
    i, j, k = 5, 7, 4
    state[4, i + 64 * (j + 12 * k)] = 0.0          # E = 0: negative thermal pressure
    for _ in range(2):
        with S.Grid(cells, length, gamma, mu0) as g:
            g.set_launch(128)
            g.upload(state)
            with pytest.raises(_lib.PamhdError) as ei:
                g.run("hlld-athena", 0.3, 0.0, 1e9, max_steps=2)
            assert ei.value.code == 2 and "(%d,%d,%d) and its -x" % (i, j, k) in str(ei.value)
            with pytest.raises(_lib.PamhdError):
                g.check()


def _launches(g, steps=5):
    """dt, flux_pass and update launches of `steps` steps (the step length is
    a launch of every step but the flat one)"""
    g.step("hlld-athena", 1e300, 0.3)
    g.enable_timing(True)
    for _ in range(steps):
        g.step("hlld-athena", 1e300, 0.3)
    n = tuple(g.kernel_time(k)[1] for k in ("dt", "flux_pass", "update"))
    ms = [g.kernel_time(k)[0] for k in ("flux_pass", "update")]
    g.enable_timing(False)
    assert min(ms) > 0
    return n


@pytest.mark.gpu
def test_kernel_timing_of_the_flat_step(gpu):
    """timing accounts the launches that untimed steps make"""
    from pamhd_amd import solver as S
    cells = (20, 9, 7)
    state, length, gamma, mu0 = _state(cells)
    with S.Grid(cells, length, gamma, mu0) as g:
        g.upload(state)
        g.timestep("hlld-athena", 0.0, 0.3)
        assert _launches(g) == (0, 5, 5)
        g.set_launch(65, 8, 4)
        assert _launches(g) == (5, 5, 5)


@pytest.mark.gpu
def test_default_step_after_setters_are_undone(gpu):
    from pamhd_amd import solver as S
    cells = (20, 9, 7)
    state, length, gamma, mu0 = _state(cells)
    flat, other = (0, 5, 5), (5, 5, 5)
    with S.Grid(cells, length, gamma, mu0) as g:
        g.upload(state)
        g.timestep("hlld-athena", 0.0, 0.3)
        for call, want in ((lambda: g.set_slabs(3), other), (lambda: g.set_slabs(1), flat),
                           (lambda: g.set_slabs(3), other), (lambda: g.set_fused_step("auto"), other),
                           (lambda: g.set_launch(128), flat), (lambda: g.set_slabs(3), other),
                           (lambda: g.set_slabs(1), flat), (lambda: g.set_launch(0, 0, 0), other),
                           (lambda: g.set_slabs(1), other), (lambda: g.set_fused_step("auto"), flat),
                           (lambda: g.set_fused_step("passes"), other), (lambda: g.set_fused_step("auto"), flat)):
            call()
            assert _launches(g) == want


@pytest.mark.gpu
def test_flat_step_replays_in_a_graph(gpu):
    """two captured steps, replayed with eager steps in between"""
    import torch
    from pamhd_amd import solver as S
    cells = (33, 7, 5)
    state, length, gamma, mu0 = _state(cells)
    with S.Grid(cells, length, gamma, mu0) as a, S.Grid(cells, length, gamma, mu0) as b:
        for g in (a, b):
            g.upload(state)
            g.timestep("hlld-athena", 0.0, 0.3)
            g.step("hlld-athena", 1e300, 0.3)
            g.step("hlld-athena", 1e300, 0.3)
        graph = torch.cuda.CUDAGraph()
        side = torch.cuda.Stream()
        with torch.cuda.graph(graph, stream=side):
            for _ in range(2):
                a.step("hlld-athena", 1e300, 0.3, sync=False, stream=side.cuda_stream)
        for rep in range(4):
            graph.replay()
            torch.cuda.synchronize()
            for _ in range(2):
                b.step("hlld-athena", 1e300, 0.3)
            np.testing.assert_array_equal(a.download(), b.download())
            if rep == 1:
                for _ in range(2):
                    assert a.step("hlld-athena", 1e300, 0.3) == b.step("hlld-athena", 1e300, 0.3)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["passes", "accumulate"])
def test_replayed_marches_between_flat_steps(gpu, mode):
    """two captured steps of another structure, replayed with eager flat
    steps in between: the flat steps' lagged length follows the replay"""
    import torch
    from pamhd_amd import solver as S
    cells = (33, 7, 5)
    state, length, gamma, mu0 = _state(cells)
    with S.Grid(cells, length, gamma, mu0) as a, S.Grid(cells, length, gamma, mu0) as b:
        for g in (a, b):
            g.set_fused_step(mode)
            g.upload(state)
            g.timestep("hlld-athena", 0.0, 0.3)
            g.step("hlld-athena", 1e300, 0.3)
        graph = torch.cuda.CUDAGraph()
        side = torch.cuda.Stream()
        with torch.cuda.graph(graph, stream=side):
            for _ in range(2):
                a.step("hlld-athena", 1e300, 0.3, sync=False, stream=side.cuda_stream)
        a.set_launch(128)
        for rep in range(4):
            for _ in range(2):
                assert a.step("hlld-athena", 1e300, 0.3) == b.step("hlld-athena", 1e300, 0.3)
            graph.replay()
            torch.cuda.synchronize()
            for _ in range(2):
                b.step("hlld-athena", 1e300, 0.3)
            np.testing.assert_array_equal(a.download(), b.download())


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["launches", "graph", "persistent"])
def test_box_cells_by_flat_index(gpu, mode):
    """solar-wind boxes with their default blocks of 256 consecutive cells,
    cells a multiple of a block, a few more and a few less, against the oracle"""
    from pamhd_amd.swbox import Ensemble
    from test_gpu_swbox import _test_box
    boxes = [_test_box(cells=c, seed=3 + q) for q, c in enumerate([(8, 8, 8), (11, 31, 9), (5, 17, 6), (9, 9, 19)])]
    refs = []
    for sb in boxes:
        ob = O.Box(sb)
        r = ob.init()
        st, steps, t = ob.run(O.HLL, 0.3, 0.0, 1e30, r, max_steps=5)
        assert st == 0 and steps == 5
        refs.append(r)
    with Ensemble(boxes) as e:
        e.timestep("hll-athena", 0.0, 0.3)
        print(mode, flush=True)
        e.run("hll-athena", 0.3, 5, use_graph=mode == "graph", persistent=mode == "persistent")
        e.check()
        for q, r in enumerate(refs):
            np.testing.assert_array_equal(e.download(q), r, err_msg="box %d" % q)


@pytest.mark.gpu
@pytest.mark.parametrize("cells", [(2, 3, 900), (2, 3, 1200), (65, 5, 4), (1, 1, 65535), (32, 32, 17),
                                   (32, 32, 1), (41, 25, 1)])
def test_substep_preparation_paths(gpu, cells):
    """substepped steps of grids around the limits of the one-block
    preparation (16384 cells, 1024 blocks of 64 x 4 cells; 1024 cells for its
    restriction of the levels) and with the most
    planes a launch has (no plane of blocks past them), against the oracle"""
    from pamhd_amd import configs
    from pamhd_amd import solver as S
    state, length, gamma, mu0 = configs.hot_blob(cells, contrast=30.0, radius=0.3, seed=3)
    ref = state.copy()
    og = O.make_grid(cells, length, gamma, mu0)
    st, steps, t, largest = O.run_periodic_substep(og, O.HLLD, 0.3, 0, 999, 0.0, 1e9, ref, max_steps=3)
    assert st == 0 and largest == 4
    with S.Grid(cells, length, gamma, mu0) as g:
        g.upload(state)
        g.set_substepping(0, 999)
        print("cells", cells, flush=True)
        assert g.run("hlld-athena", 0.3, 0.0, 1e9, max_steps=3) == (steps, t)
        assert g.last_max_substep() == largest
        np.testing.assert_array_equal(g.download(), ref)
