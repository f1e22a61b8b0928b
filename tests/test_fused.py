"""The fused engines (default of the 2D models) where it can go wrong: grids at the
edges of its strips (64 - 2S owned columns, partial strips), rows narrower than a wave, runs
that end in launches of fewer steps, materials with and without classes, boundary classes with
several entries and more classes than a tile holds.  FP64 against the oracle bit for bit, the
FP32 forms against the LDS-tile engine's bits."""
import numpy as np
import pytest

import pyfds_amd
import pyfds_amd.batch
import scenes

pytestmark = pytest.mark.gpu

STEPS = 23      # three launches of six stages and one of five; six of four, one of three


def _scene(model, nx, ny, steps=STEPS, medium='block', boundaries='plain', seed=0, ratio=1.0,
           mu=0.0):
    rng = np.random.default_rng(seed)
    n = nx * ny
    thermal = model.startswith('Thermal')
    dx = 1e-3 if thermal else 1e-4
    kwargs = dict(x_samples=nx, x_delta=dx, y_samples=ny, y_delta=dx * ratio, t_samples=steps)
    if thermal:
        kind, base = 'ThermalMaterial', dict(heat_capacity=4000.0, density=1000.0,
                                             thermal_conductivity=0.6)
        kwargs['t_delta'] = 0.1 * dx ** 2 * 4e6 / 50.0
        main, other = 'temperature', ('heat_flux_x', 'heat_flux_y')
    else:
        kind, base = 'AcousticMaterial', dict(scenes.WATER, absorption_coef=mu)
        kwargs['t_delta'] = 0.4 * dx / 5900.0
        main, other = 'pressure', ('velocity_x', 'velocity_y')

    def material(i):
        if thermal:
            return kind, dict(base, thermal_conductivity=1.0 + i % 50)
        return kind, dict(base, sound_velocity=1000.0 + 7.0 * i, density=900.0 + 3.0 * i)

    if medium == 'block':
        cells = np.flatnonzero(rng.random(n) < 0.3)
        regions = [(cells, material(11))] if cells.size else []
    else:               # one material a row: more classes than the kernels hold (64) if ny > 63
        regions = [(np.arange(r * nx, (r + 1) * nx), material(r)) for r in range(ny)]
    signal = rng.standard_normal(steps)
    point = [int(rng.integers(n))]
    bounds = {main: [dict(indices=point, value=signal, additive=True)]}
    if boundaries != 'plain':
        x, y = np.arange(nx), np.arange(ny)
        bounds[other[0]] = [dict(indices=np.concatenate([y * nx, y * nx + nx - 1]), value=0.0,
                                 additive=False)]
        bounds[other[1]] = [dict(indices=np.concatenate([x, x + (ny - 1) * nx]), value=0.25,
                                 additive=False)]
        # chains of entries: the same cells again, and a repeated index
        bounds[main] += [dict(indices=point * 2, value=0.5, additive=True),
                         dict(indices=[0, n - 1, point[0]], value=signal[::-1].copy(),
                              additive=True)]
    if boundaries == 'many':      # a signal a point, two rows of them: more than a tile holds
        k = 2 * nx
        bounds[main].append(dict(indices=list(range(k)),
                                 value=[rng.standard_normal(steps) for _ in range(k)],
                                 additive=True))
    outs = [int(v) for v in rng.integers(0, n, size=6)]
    return dict(name='fused', model=model, kwargs=kwargs, material=(kind, base), regions=regions,
                init={main: rng.standard_normal(n)}, boundaries=bounds,
                outputs={main: [outs, list(range(min(n, 130)))], other[0]: [outs],
                         other[1]: [outs]},
                plan=[('simulate', steps - 10), ('simulate', 7), ('simulate', 3)])


def _run(scene, **attrs):
    fld = scenes.build_field(pyfds_amd, pyfds_amd.regions, scene)
    for k, v in attrs.items():
        setattr(fld, k, v)
    scenes.run_plan(fld, scene)
    res = scenes.collect(fld, scene)
    group = fld._runner().lib.fds_steps_per_launch(fld._runner().ctx)
    fld._runner().close()
    return res, group


CASES = [
    ('Acoustic2D', 52, 40, 'block', 'plain', 1.0, 0),      # one column block (4 stages: 56)
    ('Acoustic2D', 57, 9, 'block', 'walls', 1.0, 0),       # one column more; partial strip
    ('Acoustic2D', 113, 70, 'rows', 'walls', 1.25, 7),     # coefficients cell by cell
    ('Acoustic2D', 1, 50, 'block', 'plain', 1.0, 0),
    ('Acoustic2D', 3, 33, 'block', 'walls', 1.0, 5),
    ('Acoustic2D', 200, 2, 'block', 'plain', 1.25, 0),
    ('Acoustic2D', 520, 510, 'block', 'walls', 1.0, 0),    # six stages a launch
    ('Acoustic2D', 130, 60, 'block', 'many', 1.0, 16),     # leaves the engine
    ('Acoustic3DAxi', 105, 66, 'rows', 'walls', 1.0, 4),
    ('Acoustic3DAxi', 521, 511, 'block', 'plain', 1.0, 0),
    ('Thermal2D', 64, 31, 'block', 'walls', 1.0, 0),
    ('Thermal2D', 530, 500, 'rows', 'walls', 1.25, 0),
    ('Thermal3DAxi', 71, 65, 'rows', 'plain', 1.0, 9),
    ('Thermal3DAxi', 517, 513, 'block', 'walls', 1.0, 0),
]


@pytest.mark.parametrize('model,nx,ny,medium,boundaries,ratio,strip', CASES)
def test_fp64_matches_oracle_bitwise(model, nx, ny, medium, boundaries, ratio, strip):
    scene = _scene(model, nx, ny, medium=medium, boundaries=boundaries, ratio=ratio)
    print('fused', model, nx, ny, medium, boundaries, flush=True)
    ref = scenes.run_oracle(scene)
    got, group = _run(scene, strip_height=strip)
    assert group == (2 if boundaries == 'many' else 6 if nx * ny >= 1 << 18 else 4)
    for k in ref:
        np.testing.assert_array_equal(got[k], ref[k], err_msg=k)


@pytest.mark.parametrize('form', ['fp32', 'fp32_kahan'])
@pytest.mark.parametrize('case', [2, 6, 8, 11, 13])
def test_fp32_forms_equal_tile_engine(case, form):
    model, nx, ny, medium, boundaries, ratio, strip = CASES[case]
    scene = _scene(model, nx, ny, medium=medium, boundaries=boundaries, ratio=ratio, seed=3)
    print('fused', form, model, nx, ny, flush=True)
    a, _ = _run(scene, form=form, tile=1)
    b, _ = _run(scene, form=form, strip_height=strip)
    for k in a:
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)


# lossy: one, two or three stages a launch, one more ghost column on the right, twice the ghost
# rows below
LOSSY = [
    ('Acoustic2D', 57, 40, 'block', 'plain', 1.0, 0),
    ('Acoustic2D', 58, 9, 'block', 'walls', 1.0, 0),
    ('Acoustic2D', 115, 70, 'block', 'walls', 1.25, 7),
    ('Acoustic2D', 1, 50, 'block', 'plain', 1.0, 0),
    ('Acoustic2D', 2, 33, 'block', 'walls', 1.0, 5),
    ('Acoustic2D', 200, 2, 'block', 'plain', 1.25, 0),
    ('Acoustic2D', 90, 71, 'rows', 'walls', 1.0, 0),       # too many classes: one step a launch
    ('Acoustic2D', 130, 60, 'block', 'many', 1.0, 16),     # leaves the engine
    ('Acoustic3DAxi', 106, 66, 'block', 'walls', 1.0, 4),
    ('Acoustic3DAxi', 171, 90, 'block', 'walls', 1.25, 0),
    ('Acoustic3DAxi', 64, 40, 'rows', 'plain', 1.0, 0),    # forty classes
    ('Acoustic2D', 530, 500, 'block', 'walls', 1.0, 0),
]


@pytest.mark.parametrize('model,nx,ny,medium,boundaries,ratio,strip', LOSSY)
def test_fp64_lossy_matches_oracle_bitwise(model, nx, ny, medium, boundaries, ratio, strip):
    scene = _scene(model, nx, ny, medium=medium, boundaries=boundaries, ratio=ratio, mu=0.3)
    print('fused lossy', model, nx, ny, medium, boundaries, flush=True)
    ref = scenes.run_oracle(scene)
    got, group = _run(scene, strip_height=strip)
    assert (group > 1) == (boundaries != 'many' and (medium, ny) != ('rows', 71))
    for k in ref:
        np.testing.assert_array_equal(got[k], ref[k], err_msg=k)


@pytest.mark.parametrize('form', ['fp32', 'fp32_kahan'])
@pytest.mark.parametrize('case', [2, 4, 9, 11])
def test_fp32_lossy_forms_equal_tile_engine(case, form):
    model, nx, ny, medium, boundaries, ratio, strip = LOSSY[case]
    scene = _scene(model, nx, ny, medium=medium, boundaries=boundaries, ratio=ratio, seed=3,
                   mu=0.3)
    print('fused lossy', form, model, nx, ny, flush=True)
    a, _ = _run(scene, form=form, tile=1)
    b, _ = _run(scene, form=form, strip_height=strip)
    for k in a:
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)


def _batch_scenes(models):
    sizes = [(130, 61), (57, 200), (300, 40), (3, 70), (515, 520)]
    return [_scene(m, *sizes[i], medium='block', boundaries='walls' if i % 2 else 'plain',
                   ratio=r, seed=i) for i, (m, r) in enumerate(models)]


@pytest.mark.parametrize('models', [
    [('Acoustic2D', 1.0), ('Acoustic3DAxi', 1.0), ('Acoustic3DAxi', 1.25), ('Acoustic2D', 1.0),
     ('Acoustic2D', 1.0)],
    [('Acoustic2D', 1.25), ('Thermal2D', 1.0), ('Thermal3DAxi', 1.0), ('Thermal2D', 1.25)]])
def test_fp64_batch_matches_oracle_bitwise(models):
    """Batches on the fused engine: six and four stages a launch, remainders in one launch; then
    a boundary list that no longer fits it, which moves the batch to its streaming shape."""
    built = [(sc, scenes.build_field(pyfds_amd, pyfds_amd.regions, sc))
             for sc in _batch_scenes(models)]
    fields = [f for _, f in built]
    batch = pyfds_amd.batch.BatchRunner(fields, chunk=8)
    for n in (13, 7):
        batch.simulate(n)
    group = batch.lib.fds_batch_steps_per_launch(batch.handle)
    assert group == (6 if sum(f.num_points for f in fields) >= 1 << 18 else 4)
    more = [dict(indices=list(range(250)), value=[np.full(STEPS, 0.1 * i) for i in range(250)],
                 additive=True)]
    main = next(iter(built[0][0]['boundaries']))
    getattr(fields[0], main).add_boundary(pyfds_amd.regions.Region(more[0]['indices']),
                                          value=more[0]['value'], additive=True)
    batch.simulate(3)
    assert batch.lib.fds_batch_steps_per_launch(batch.handle) == 2
    for i, (sc, fld) in enumerate(built):
        print('member', i, sc['model'], flush=True)
        o = scenes.build_oracle(sc)
        o.simulate(20)
        if i == 0:
            o.boundaries[main] = o.boundaries[main] + more
        o.simulate(3)
        got = scenes.collect(fld, sc)
        for comp in scenes.COMPONENTS[sc['model']]:
            np.testing.assert_array_equal(got['values/' + comp], o.components[comp],
                                          err_msg='%d %s' % (i, comp))
            for k, out in enumerate(o.outputs[comp]):
                np.testing.assert_array_equal(got['signals/%s/%d' % (comp, k)],
                                              np.array(out['signals'], dtype=float),
                                              err_msg='%d %s' % (i, comp))


@pytest.mark.parametrize('mu', [0.0, 0.3])
def test_boundary_cells_without_entries_do_nothing(mu):
    """``fds_set_boundaries`` takes cells with no entry, first, between others and last of a tile,
    of every component: the tile engine's bits."""
    nat = pyfds_amd._native
    nx, ny, steps = 90, 40, 11
    signal = np.random.default_rng(5).standard_normal(steps)
    table = np.concatenate([[0.5, -0.25], signal])
    inf = np.iinfo(np.int64).max
    entry = {'set': (0.0, 0, 0, inf), 'add': (1.0, 1, 0, inf), 'signal': (1.0, 2, 1, steps)}
    programs = [  # component 0, 1, 2: (cell, entries)
        [(3, []), (40, ['set']), (41, []), (nx + 7, ['signal', 'add']), (9 * nx + 2, []),
         (30 * nx + 60, ['add']), (39 * nx + 89, [])],
        [(5, ['add']), (nx + 6, []), (20 * nx + 61, [])],
        [(0, []), (17 * nx, []), (39 * nx + 88, [])]]
    res = []
    for tile in (1, -1):
        print('empty programs', mu, tile, flush=True)
        fld = scenes.build_field(pyfds_amd, pyfds_amd.regions, _scene('Acoustic2D', nx, ny, mu=mu))
        fld.tile = tile
        fld.assemble_matrices()
        run = fld._runner()
        run.sync(fld)
        for k, prog in enumerate(programs):
            ents = [entry[e] for _, es in prog for e in es]
            cells = nat.i64([c for c, _ in prog])
            ptr = np.concatenate([[0], np.cumsum([len(es) for _, es in prog])]).astype(np.int32)
            a = nat.f64([e[0] for e in ents])
            off, stride, length = (nat.i64([e[i] for e in ents]) for i in (1, 2, 3))
            nat.check(run.lib.fds_set_boundaries(
                run.ctx, k, cells.size, nat.lptr(cells), nat.iptr(ptr), len(ents), nat.dptr(a),
                nat.lptr(off), nat.lptr(stride), nat.lptr(length), table.size, nat.dptr(table)))
        nat.check(run.lib.fds_run(run.ctx, 0, steps, 0))
        res.append([run.download(k) for k in range(3)])
        run.close()
    for a, b in zip(*res):
        np.testing.assert_array_equal(a, b)


def _signals_scene(nx, ny, cells, seed=0):
    """A signal of its own on each of ``cells``, on top of the plain scene."""
    sc = _scene('Acoustic2D', nx, ny, seed=seed)
    rng = np.random.default_rng(seed)
    sc['boundaries']['pressure'] = [dict(indices=list(cells), additive=True,
                                         value=[rng.standard_normal(STEPS) for _ in cells])]
    return sc


@pytest.mark.parametrize('count', [63, 64])
def test_as_many_boundary_classes_as_a_tile_holds(count):
    scene = _signals_scene(50, 8, range(3, 3 + 5 * count, 5))
    print('classes', count, flush=True)
    ref = scenes.run_oracle(scene)
    got, group = _run(scene, strip_height=8)
    assert group == (4 if count == 63 else 2)
    for k in ref:
        np.testing.assert_array_equal(got[k], ref[k], err_msg=k)


def test_strips_too_tall_for_the_classes_leave_other_heights_alone():
    """Two signals a row: strips of 48 rows see more classes than a tile holds, strips of 8 and the
    height of the grid's own choice do not, whatever was tried before."""
    nx, ny = 130, 60
    scene = _signals_scene(nx, ny, [r * nx + c for r in range(ny) for c in (20, 21)])
    fld = scenes.build_field(pyfds_amd, pyfds_amd.regions, scene)
    fld.assemble_matrices()
    run = fld._runner()
    run.sync(fld)
    lib = run.lib

    def go(n, strip=None, tile=None):
        if tile is not None:
            pyfds_amd._native.check(lib.fds_set_tile(run.ctx, tile))
        if strip is not None:
            pyfds_amd._native.check(lib.fds_set_strip_height(run.ctx, strip))
        fld.simulate(n)
        return lib.fds_steps_per_launch(run.ctx)

    groups = [go(3, 48), go(3, 8), go(3, 48), go(2, 0), go(1, 48), go(2, 0, 1), go(2, 0, -1)]
    fld.assemble_matrices()
    groups += [go(2, 48), go(2, 8)]
    assert groups == [2, 4, 2, 4, 2, 1, 4, 2, 4]
    ref = scenes.build_oracle(scene)
    ref.simulate(20)
    np.testing.assert_array_equal(fld.pressure.values, ref.components['pressure'])


def test_autotuner_times_the_engine_a_field_runs_by_itself(tmp_path, monkeypatch):
    """By default tile -1 is among the candidates, of single fields and batches, and picks stored
    before it was one are not applied."""
    from pyfds_amd import autotune
    monkeypatch.setattr(autotune, 'CACHE', str(tmp_path / 'tune.json'))
    fields = [scenes.build_field(pyfds_amd, pyfds_amd.regions, _scene('Acoustic2D', 90, 40, seed=i))
              for i in range(2)]
    for f in fields:
        f.assemble_matrices()
    old = autotune._key(fields[:1]).rsplit('|', 1)[0] + '|v4'
    autotune._save_cache({old: dict(tile=0, strip=0, chunk=50, table={'0,0,50': 1.0})})
    tile, _, table = autotune.tune_field(fields[0], steps=6)
    assert '-1,0,50' in table and '-1,8,50' in table and '0,0,50' in table
    assert fields[0].tile == tile
    _, _, table = autotune.tune_batch(fields, steps=6, use_cache=False)
    assert '-1,0,50' in table
    tile, _, table = autotune.tune_field(fields[0], steps=6, default_engine=False)
    assert tile >= 0 and '-1,0,50' not in table


@pytest.mark.parametrize('mu', [0.0, 0.3])
@pytest.mark.parametrize('rows', [62, 63, 64])
def test_as_many_materials_as_the_table_holds(rows, mu):
    """A material a row; the class table holds 63.  Lossy fields of more take one step a launch."""
    scene = _scene('Acoustic2D', 71, rows, medium='rows', mu=mu)
    print('materials', rows, mu, flush=True)
    ref = scenes.run_oracle(scene)
    got, group = _run(scene)
    assert group == (4 if not mu else 3 if rows <= 63 else 1)
    for k in ref:
        np.testing.assert_array_equal(got[k], ref[k], err_msg=k)


@pytest.mark.parametrize('form', ['fp64', 'fp32'])
def test_classes_of_scattered_materials(form):
    """50 materials cell by cell at random, a few of them equal in all but one coefficient."""
    scene = _scene('Acoustic2D', 301, 97, seed=9)
    rng = np.random.default_rng(9)
    of = rng.integers(0, 50, 301 * 97)
    base = dict(scenes.WATER)
    scene['regions'] = [(np.flatnonzero(of == i), ('AcousticMaterial', dict(
        base, sound_velocity=1000.0 + 40.0 * (i // 2), density=900.0 + (i % 2)))) for i in range(50)]
    a, _ = _run(scene, form=form, tile=1)
    b, group = _run(scene, form=form)
    assert group == 4
    for k in a:
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)


@pytest.mark.parametrize('nx, ny', [(130, 60), (5, 90)])
def test_boundary_and_output_cells_in_any_order(nx, ny):
    """Cells handed over in descending and in random order (the event lists are sorted by tile and
    place), rows shorter than a strip among them: the oracle's bits."""
    scene = _scene('Acoustic2D', nx, ny, boundaries='walls', seed=2)
    rng = np.random.default_rng(2)
    n = nx * ny
    scene['boundaries']['velocity_x'].append(dict(
        indices=[int(v) for v in rng.permutation(n)[:n // 3]], value=0.125, additive=False))
    scene['boundaries']['velocity_y'].append(dict(
        indices=list(range(n - 1, 0, -7)), value=-0.5, additive=True))
    scene['outputs']['pressure'].append([int(v) for v in rng.permutation(n)[:400]])
    scene['outputs']['velocity_y'].append(list(range(n - 1, 0, -11)))
    ref = scenes.run_oracle(scene)
    got, group = _run(scene)
    assert group == 4
    for k in ref:
        np.testing.assert_array_equal(got[k], ref[k], err_msg=k)


@pytest.mark.parametrize('model, form, nx, ny, group', [
    ('Acoustic2D', 'fp32', 1031, 1021, 4), ('Acoustic2D', 'fp32_kahan', 1033, 1019, 4),
    ('Acoustic2D', 'fp64', 1031, 1021, 3), ('Acoustic3DAxi', 'fp64', 2053, 2047, 3)])
def test_large_lossy_fields_equal_tile_engine(model, form, nx, ny, group):
    """The stage counts that only large lossy fields take, with remainder launches."""
    scene = _scene(model, nx, ny, boundaries='walls', mu=0.3, seed=6)
    scene['plan'] = [('simulate', 9), ('simulate', 6)]
    print('large lossy', model, form, flush=True)
    a, _ = _run(scene, form=form, tile=1)
    b, got = _run(scene, form=form)
    assert got == group
    for k in a:
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)
