"""Prefill with 8 and 16 key splits, merged by a second launch (few query
blocks over many keys): forced counts that leave splits empty, and the counts
the split rule takes for a short batch after a long history, each against the
oracle at the path's 2e-3 x RMS bar, repeated bit for bit."""
import numpy as np
import pytest

from helpers import TOL, rel_err
from test_attn_hostemu import Emu, built  # noqa: F401  (built: the emulator's build)


@pytest.mark.parametrize("splits", [8, 16])
def test_forced_on_the_emulated_machine(built, tmp_path, splits):  # noqa: F811
    e = Emu(tmp_path, H=4, Hkv=1, max_context=640, window=64)
    e.prefill(5, 0, 330)
    e.prefill(0, 0, 40)       # two tiles: most splits empty
    launches = e.run(G3ATTN_PREFILL_SPLITS=splits)
    assert launches["prefill_merge_kernel"][0] == 2, launches


@pytest.mark.gpu
@pytest.mark.parametrize("splits", [8, 16])
def test_forced_split_counts(monkeypatch, splits):
    from test_gpu_prefill import PrefillCase, _check_cache, _ctx

    monkeypatch.setenv("G3ATTN_PREFILL_SPLITS", str(splits))
    cases = [PrefillCase(74, layer=3, start_pos=1500, n=700, max_context=4096),
             PrefillCase(75, layer=5, start_pos=0, n=2048, max_context=4096),
             PrefillCase(76, layer=5, start_pos=0, n=17, max_context=4096)]
    with _ctx(max_context=4096, num_layers=12) as c:
        for i, case in enumerate(cases):
            got = case.gpu(c)
            assert c.last_splits(1) == splits, (i, c.last_splits(1))
            want, Kc, Vc = case.oracle()
            err = rel_err(got, want)
            print(f"[forced splits {splits} case {i}] rel_err={err:.3e}", flush=True)
            assert err <= TOL, (splits, i, err)
            _check_cache(c, case, Kc, Vc)


@pytest.mark.gpu
def test_the_rule_takes_them_after_a_long_history():
    from test_gpu_prefill import PrefillCase, _ctx

    case = PrefillCase(77, layer=5, start_pos=3300, n=33, max_context=4096)
    with _ctx(max_context=4096, num_layers=12) as c:
        got = case.gpu(c)
        assert c.last_splits(1) in (8, 16)
        want, _, _ = case.oracle()
        assert rel_err(got, want) <= TOL
        assert np.array_equal(got, case.gpu(c))
