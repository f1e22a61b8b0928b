"""The benchmark's line: the contract's keys, JSON, short enough to be read back whole."""
import importlib.util
import json
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_summary_keeps_the_contract_and_stays_short():
    spec = importlib.util.spec_from_file_location('bench', os.path.join(ROOT, 'bench.py'))
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    table = {'%d,%d,50' % (t, h): 123.45 for t in range(-1, 21) for h in range(6)}
    form = dict(value=1234.567, ms_per_step=0.0123, kernel_us=12.34, autotune=dict(table=table),
                rel_l2_vs_fp64=1.3543455021928995e-07)
    forms = {f: dict(form) for f in ('fp64', 'fp32', 'fp32_kahan')}
    cpu = dict(value=0.07457, unit='Gcell-updates/s', cores=1, kind='port', sample='x' * 300,
               host=dict(model='y' * 100))
    line = dict(metric=bench.METRIC, value=345.678, unit='Gcell-updates/s', n_gpus=1, steps=20,
                warmup=5, ms_per_step=0.0127, higher_is_better=True, scaling='weak',
                vs_baseline=None, dtype='f64', data='synthetic',
                config=dict(workload='w' * 110, nx=2048, ny=2048, form='fp64', recorded_points=64),
                roofline=dict(bound='hbm', achieved=5802.2, peak=8000.0, unit='GB/s', frac=0.7253,
                              traffic=235064416, basis='z' * 200),
                roofline_detail=dict(note='n' * 500), cpu_baseline=cpu,
                cpu_baseline_all_cores=dict(cpu), forms=forms,
                lossy=dict(forms, config='c'), batched=dict(forms, config='c', cpu_baseline=cpu),
                thermal2d=dict(forms, config='c', cpu_baseline=cpu),
                acoustic1d=dict(default=dict(us_per_step=0.352), fp64=dict(us_per_step=0.352)),
                learned_bc=dict(reflected_energy=0.000466, learned_s=0.045, enlarged_s=0.07,
                                speedup_vs_enlarged=1.553, training=dict(loss=[[0, 1.0]] * 9),
                                default_engines=dict(learned_s=0.0157, enlarged_s=0.0155,
                                                     speedup_vs_enlarged=0.984)))
    text = json.dumps(bench.summary(line, '/tmp/detail.json'))
    assert len(text) < 2000 and '\n' not in text
    got = json.loads(text)
    for k in ('metric', 'value', 'unit', 'n_gpus', 'steps', 'warmup', 'ms_per_step',
              'higher_is_better', 'scaling', 'vs_baseline', 'dtype', 'data', 'config'):
        assert got[k] == line[k]
    line = {k: v for k, v in line.items() if k not in ('lossy', 'acoustic1d', 'learned_bc')}
    line['cpu_baseline'] = None
    bench.summary(line, 'd')          # sections left out
