"""Prefill with 8 and 16 key splits, merged by a second launch (few query
blocks over many keys): forced counts that leave splits empty, and the counts
the split rule takes for a short batch after a long history, each against the
oracle at the path's 2e-3 x RMS bar, repeated bit for bit; and the same counts
inside the whole model's batched prefill, where the merge writes o_proj's bf16
planes, against the token forward."""
import numpy as np
import pytest

from helpers import TOL, rel_err
from test_attn_hostemu import Emu, _emu_for, _forward_model, built  # noqa: F401  (built: the emulator's build)
from test_gemm_forms import G, random_model


@pytest.mark.parametrize("splits", [8, 16])
def test_forced_on_the_emulated_machine(built, tmp_path, splits):  # noqa: F811
    e = Emu(tmp_path, H=4, Hkv=1, max_context=640, window=64)
    e.prefill(5, 0, 330)
    e.prefill(0, 0, 40)       # two tiles: most splits empty
    launches = e.run(G3ATTN_PREFILL_SPLITS=splits)
    assert launches["prefill_merge_kernel"][0] == 2, launches


def test_the_rules_empty_splits_fetch_nothing_out_of_range(built, tmp_path):  # noqa: F811
    """16 tokens at position 2035 are 65 key tiles, which the rule deals to 16
    splits five at a time: three of them get none.  The emulated machine stops
    a buffer access whose scalar offset passes the buffer's end."""
    e = Emu(tmp_path, H=1, Hkv=1, max_context=2056, window=64)
    e.kv_append(5, 0, 2035)
    e.prefill(5, 2035, 16)
    launches = e.run()
    assert launches["prefill_kernel"] == (1, 16) and launches["prefill_merge_kernel"][0] == 1, launches


def test_fewer_splits_where_memory_is_short(built, tmp_path):  # noqa: F811
    """The same call on a device whose largest allocation holds the staged
    keys and four splits' parts, but not sixteen's."""
    e = Emu(tmp_path, H=1, Hkv=1, max_context=2056, window=64)
    e.kv_append(5, 0, 2035)
    e.prefill(5, 2035, 16)
    staged = 2112 * 256 * 2 * 4
    launches = e.run(HOSTEMU_MALLOC_MAX=staged + 8 * 16 * 256 * 4)
    assert launches["prefill_kernel"] == (1, 4) and "prefill_merge_kernel" not in launches, launches


@pytest.mark.parametrize("splits", [4, 8])
def test_profiled_time_covers_the_merge(built, tmp_path, splits):  # noqa: F811
    """g3attn_profile_read's kind 1 is the time to the finished output on
    either side of four splits: the merge is inside the kernel up to four, and
    its own launch beyond."""
    e = Emu(tmp_path, H=1, Hkv=1, max_context=640, window=64)
    e.lines.append("profile 1")
    e.prefill(5, 0, 400)
    e.lines.append("profile 1")
    e.run(G3ATTN_PREFILL_SPLITS=splits)
    ms = {ln.split()[1].strip("()").split("<")[0]: float(ln.split()[-1]) for ln in e.stdout.splitlines()
          if ln.startswith("launch prefill_") or ln.startswith("launch (prefill_")}
    profiled = [ln.split()[1:] for ln in e.stdout.splitlines() if ln.startswith("profile ")]
    assert len(ms) == (2 if splits > 4 else 1), ms
    assert profiled[0][0] == "1" and int(profiled[0][2]) == 1
    assert float(profiled[0][1]) >= sum(ms.values()) - 0.2, (profiled, ms)


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


@pytest.mark.parametrize("splits", [8, 16])
def test_planes_on_the_emulated_machine(built, tmp_path, splits):  # noqa: F811
    """Two chunks through the small model, the second after history, with the
    merge writing the attention output as planes in every layer: the last
    token's logits at the token forward's 1e-4 x RMS."""
    f, embed, layers, norm, tokens, want = _forward_model(32)
    e = _emu_for(tmp_path, f)
    e.model(embed, layers, norm)
    e.lines.append("upload")
    e._save("a.bin", tokens[:16].astype(np.int32))
    e._save("b.bin", tokens[16:].astype(np.int32))
    e.logits("prefill_tokens", "16 a.bin 0", want[15], "first chunk")
    e.logits("prefill_tokens", "16 b.bin 16", want[31], "second chunk")
    launches = e.run(G3ATTN_PREFILL_SPLITS=splits)
    assert launches["prefill_merge_kernel"][0] == 2 * f["layers"], launches


@pytest.mark.gpu
@pytest.mark.parametrize("start,n,forced", [(947, 77, None), (4000, 64, None), (300, 40, 8), (300, 40, 16)])
def test_planes_in_the_model(monkeypatch, start, n, forced):
    """A follow-up chunk through six layers (five local, one global), at the
    rule's own 8 or 16 splits and forced ones, against the token forward over
    the same chunk on the same history, at 1e-4 x RMS (2e-6 measured)."""
    if forced:
        monkeypatch.setenv("G3ATTN_PREFILL_SPLITS", str(forced))
    rng = np.random.default_rng(start + n)
    HW, keep = random_model(rng, 256, 512, 96, 6)
    tokens = rng.integers(0, 96, start + n).astype(np.int32)
    cfg = G.default_config(num_layers=6, hidden_size=256, intermediate_size=512, vocab_size=96, max_context=4096)
    with G.Context(cfg, 4096) as ctx:
        ctx.upload_weights(HW)
        ctx.prefill_tokens(tokens[:start], logits=False)
        got = ctx.prefill_tokens(tokens[start:], start_pos=start)
        assert ctx.last_splits(1) in ((forced,) if forced else (8, 16)), ctx.last_splits(1)
    with G.Context(cfg, 4096) as ctx:
        ctx.upload_weights(HW)
        ctx.prefill_tokens(tokens[:start], logits=False)
        for i in range(start, start + n):
            want = ctx.forward_token(tokens[i], i)
    e = rel_err(got, want)
    print(f"[planes start={start} n={n} forced={forced}] {e:.2e}", flush=True)
    assert e <= 1e-4
