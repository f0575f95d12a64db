"""The forms of the batched projection (csrc/gemm.hip) and the rule that picks
them, at the sizes where each can go wrong: the token counts on either side of
a form's limit, weight rows that end inside a workgroup's, K that ends with
half a 64-wide chunk, one chunk alone, and split sums.

- On the CPU the rule itself (g3k_gemm_plan): what it gives is accepted by
  the launcher for every size the entry points take, and the split products
  stay inside a bounded workspace.
- On the CPU the kernels' own source on the emulated machine, and on the GPU
  the built ones, against fp64: |C - C64| <= (2^-16 + K 2^-24) sum_k |w_k x_k|
  per element (the hi / lo split of X, 2^-17, doubled; fp32 accumulation in
  any order).  The GEGLU forms run in the batched prefills of
  test_gpu_gemm.py (40 tokens) and test_gpu_model_full.py (192 and 2048).
"""
import ctypes as C

import numpy as np
import pytest

from helpers import DeviceBuffer, g3attn
from test_attn_hostemu import Emu, built  # noqa: F401  (built: the emulator's build)

G = g3attn()
TILE, WIDE, NARROW, QUAD128, QUAD256 = range(5)


def plan(N, K, M, geglu=0, consumer_adds=0, n_cu=256):
    kind, s = C.c_int(), C.c_int()
    m = (C.c_int * len(M))(*M)
    G.lib().g3k_gemm_plan(N, K, len(M), m, geglu, consumer_adds, n_cu, C.byref(kind), C.byref(s))
    return kind.value, s.value


@pytest.mark.parametrize("K", [32, 64, 96, 2048, 2592, 10240])
def test_plan_stays_in_the_launchers_limits(K):
    rng = np.random.default_rng(K)
    Ns = [1, 15, 16, 17, 32, 33, 64, 65, 128, 129, 1535, 1536, 4096, 4097, 65536, 2000000]
    for N in Ns + [int(n) for n in np.exp(rng.uniform(0, 12, 40))]:
        for M in ([4], [64], [2560], [262208], [2048, 1024, 1024], [256, 256, 256]):
            for adds in (0, 1):
                kind, s = plan(N, K, M, 0, adds)
                assert 0 <= kind <= QUAD256 and 1 <= s <= (K + 63) // 64, (N, M, kind, s)
                if kind in (NARROW, WIDE):
                    assert N <= (4096 if kind == NARROW else 128)
                if kind in (QUAD128, QUAD256):
                    assert s == 1 and not adds
                if s > 1:
                    assert 4 * s * N * sum(M) <= 256e6, (N, M, s)
        kind, s = plan(N, K, [10240, 10240], 1)
        assert 1 <= s <= (K + 63) // 64
        assert kind == (WIDE if N <= 128 else TILE)
        assert s == 1 or kind == WIDE


@pytest.mark.parametrize("N,M,K,kinds", [
    (128, 262208, 2560, (WIDE, TILE)), (100, 262208, 512, (WIDE, QUAD128, QUAD256)),   # W read once
    (100, 30000, 2560, (WIDE,)), (100, 2560, 10240, (NARROW,)), (1, 262208, 2560, (NARROW,)),
    (1024, 102400, 96, (QUAD256,)), (2048, 12368, 352, (QUAD256,)), (1024, 10240, 512, (QUAD128, QUAD256)),   # short rows
    (2048, 10240, 2560, (TILE,)), (2048, 2560, 10240, (TILE,)),
    (4097, 256, 512, (QUAD128, QUAD256))])
def test_plan_takes_the_form_measured_fastest(N, M, K, kinds):
    """Stand-alone products on either side of the rule's lines: the forms that
    are within 5% of the fastest there."""
    assert plan(N, K, [M])[0] in kinds, plan(N, K, [M])


def test_plan_splits_where_the_sums_cost_less_than_they_save():
    assert plan(1500, 2144, [5684])[1] == 1 and plan(64, 512, [256])[1] == 1
    assert plan(384, 10240, [2560])[1] > 4 and plan(77, 10240, [2560])[1] > 1


SHAPES = [(16, 64, 32), (17, 68, 96), (33, 60, 160), (65, 132, 64), (1, 4, 224), (97, 132, 352)]


@pytest.mark.parametrize("cus", [8, 256])   # few and many splits
def test_forms_on_the_emulated_machine(built, tmp_path, cus):  # noqa: F811
    e = Emu(tmp_path)
    for N, M, K in SHAPES:
        e.matmul(N, M, K)
    e.run(HOSTEMU_CUS=cus)


def test_many_tokens_on_the_emulated_machine(built, tmp_path):  # noqa: F811
    """Past the weight stream's token limit: tiles with rows and tokens that
    end inside one, and half a chunk of K at the end."""
    assert plan(4100, 96, [4])[0] not in (NARROW, WIDE)
    e = Emu(tmp_path)
    e.matmul(4100, 4, 96)
    for kind in (TILE, QUAD128, QUAD256):
        emu_gemm(e, kind, 1, 0, 132, 260, 96)
    e.run()


def test_unsplit_where_memory_is_short(built, tmp_path):  # noqa: F811
    """The split products only save time: 100 tokens into 64 rows of 2304, 18
    splits of 25 KiB beside 900 KiB of planes, run unsplit on a device whose
    largest allocation is 1 MB; with room a second launch adds them."""
    assert plan(100, 2304, [64])[1] == 18
    for room, reduces in ((1000000, 0), (1 << 40, 1)):
        d = tmp_path / str(room)
        d.mkdir()
        e = Emu(d, H=1, Hkv=1, max_context=32)
        e.matmul(100, 64, 2304)
        launches = e.run(HOSTEMU_MALLOC_MAX=room)
        assert launches.get("split_reduce_kernel", (0, 0))[0] == reduces, launches


def emu_gemm(e, kind, ksplit, geglu, N, M, K):
    """One g3k_gemm of a given form on the emulated machine, against fp64."""
    W = [(e.rng.standard_normal((M, K)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16) for _ in range(1 + geglu)]
    X = (e.rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32)
    hi = (X.view(np.uint32) & 0xFFFF0000).view(np.float32)
    lo = ((X - hi).view(np.uint32) & 0xFFFF0000).view(np.float32)
    files = [e._name(f) for f in ("W", "U", "xh", "xl", "C")]
    e._save(files[0], W[0])
    if geglu:
        e._save(files[1], W[1])
    e._save(files[2], (hi.view(np.uint32) >> 16).astype(np.uint16))
    e._save(files[3], (lo.view(np.uint32) >> 16).astype(np.uint16))
    e.lines.append(f"gemm {kind} {ksplit} {geglu} {N} {M} {K} " + " ".join(files))
    X64 = hi.astype(np.float64) + lo
    W64 = [(w.astype(np.uint32) << 16).view(np.float32).astype(np.float64) for w in W]
    # fp32 accumulation of the planes' exact products, in any order
    prod, bound = [X64 @ w.T for w in W64], [2 * K * 2.0 ** -24 * (np.abs(X64) @ np.abs(w).T) + 1e-30 for w in W64]
    want, bar = prod[0], bound[0]
    if geglu:
        g, u = prod
        gelu = 0.5 * g * (1 + np.tanh(0.7978845608028654 * (g + 0.044715 * g ** 3)))
        want = gelu * u
        # |gelu'| <= 1.13; gelu and the product in fp32; the planes' 2^-16
        bar = 1.13 * bound[0] * (np.abs(u) + bound[1]) + np.abs(gelu) * bound[1]
        bar = bar + 2.0 ** -16 * np.abs(want) + 8 * 2.0 ** -24 * np.abs(g * u)
    e.checks.append((files[4], want, f"gemm kind={kind} S={ksplit} geglu={geglu} N={N} M={M} K={K}", bar))


@pytest.mark.parametrize("fetch", ["early", "late"])
@pytest.mark.parametrize("kind,geglu,N", [(WIDE, 1, n) for n in (32, 64, 96, 128)]
                         + [(NARROW, 0, n) for n in (16, 32, 48, 64)] + [(TILE, 0, 128), (TILE, 1, 128), (QUAD128, 0, 128), (QUAD256, 0, 128)])
def test_rings_turn_over(built, tmp_path, kind, geglu, N, fetch):  # noqa: F811
    """Each form with more chunks per split than its LDS rings have slots, so
    that every slot is refilled while others are read: 11 and 12 chunks (the
    last a half one) in two splits, the tiles' gate and up 23 in one.  Late:
    a fetch lands where the kernel waits for it and no earlier, so a count
    that waits for one too few reads the slot's old chunk; and a counted wait
    may only split fetches whose issue order is fixed."""
    e = Emu(tmp_path)
    emu_gemm(e, kind, 1 if kind == TILE and geglu else 2, geglu, N, 60, 22 * 64 + 32)
    e.run(HOSTEMU_FETCH=fetch)


@pytest.mark.gpu
@pytest.mark.parametrize("N,M,K", SHAPES + [
    (32, 4, 64), (64, 260, 2592), (77, 2560, 2592), (96, 132, 10240), (128, 2560, 2080), (129, 132, 96), (7, 8, 10240), (48, 2560, 10240),
    (300, 2560, 10240), (1500, 1028, 2592), (4100, 4, 96), (4097, 260, 32), (65, 16644, 544), (128, 30000, 1056),
    (777, 16388, 96), (640, 12364, 352), (49, 30004, 2592), (80, 30004, 2592), (128, 30004, 2592)])
def test_forms(N, M, K):
    rng = np.random.default_rng(N * 7 + M * 13 + K)
    W = ((rng.standard_normal((M, K)) / 64).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    X = rng.standard_normal((N, K)).astype(np.float32)
    with G.Context(G.default_config(max_context=256, num_layers=6), 256) as ctx:
        dW, dX, dC = DeviceBuffer.of(W), DeviceBuffer.of(X), DeviceBuffer(N * M * 4)
        ctx.matmul_bf16_device(dC.ptr, dW.ptr, dX.ptr, N, M, K)
        got = dC.download(np.float32, (N, M)).astype(np.float64)
    W64, X64 = (W.astype(np.uint32) << 16).view(np.float32).astype(np.float64), X.astype(np.float64)
    bound = (2.0 ** -16 + K * 2.0 ** -24) * (np.abs(X64) @ np.abs(W64).T) + 1e-30
    ratio = float(np.max(np.abs(got - X64 @ W64.T) / bound))
    print(f"[gemm forms] N={N} M={M} K={K} plan={plan(N, K, [M])} max err / bound = {ratio:.3f}", flush=True)
    assert np.all(np.isfinite(got)) and ratio <= 1.0


@pytest.mark.gpu
def test_captured_where_the_workspace_cannot_grow():
    """A product recorded into a HIP graph after an eager call whose workspace
    holds the planes but not this one's split products: it runs unsplit instead
    of allocating under capture.  Three replays, new activations and an eager
    call of the first product before each, against fp64."""
    hip, vp = DeviceBuffer.hip(), C.c_void_p
    hip.hipStreamBeginCapture.argtypes = [vp, C.c_int]
    hip.hipStreamEndCapture.argtypes = [vp, C.POINTER(vp)]
    hip.hipGraphInstantiate.argtypes = [C.POINTER(vp), vp, vp, vp, C.c_size_t]
    hip.hipGraphLaunch.argtypes = [vp, vp]
    for f in ("hipGraphExecDestroy", "hipGraphDestroy"):
        getattr(hip, f).argtypes = [vp]
    N, M, K, small = 40, 1024, 2592, 8
    assert plan(N, K, [M])[1] * M > 4 * plan(N, K, [small])[1] * small   # its parts do not fit
    rng = np.random.default_rng(40)
    W = ((rng.standard_normal((M, K)) / 64).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    W64 = (W.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    with G.Context(G.default_config(max_context=256, num_layers=6), 256) as ctx:
        dW, dX, dC, dS = DeviceBuffer.of(W), DeviceBuffer(N * K * 4), DeviceBuffer(N * M * 4), DeviceBuffer(N * small * 4)
        stream, graph, exe = vp(ctx.stream()), vp(), vp()

        def eager():
            ctx.matmul_bf16_device(dS.ptr, dW.ptr, dX.ptr, N, small, K)
            ctx.synchronize()

        dX.upload(np.zeros((N, K), np.float32))
        eager()
        assert hip.hipStreamBeginCapture(stream, 2) == 0     # hipStreamCaptureModeRelaxed
        ctx.matmul_bf16_device(dC.ptr, dW.ptr, dX.ptr, N, M, K)
        assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
        assert hip.hipGraphInstantiate(C.byref(exe), graph, None, None, 0) == 0
        for rep in range(3):
            X = rng.standard_normal((N, K)).astype(np.float32)
            dX.upload(X)
            eager()
            assert hip.hipGraphLaunch(exe, stream) == 0
            ctx.synchronize()
            X64 = X.astype(np.float64)
            bound = (2.0 ** -16 + K * 2.0 ** -24) * (np.abs(X64) @ np.abs(W64).T)
            for buf, m in ((dC, M), (dS, small)):
                got = buf.download(np.float32, (N, m)).astype(np.float64)
                assert np.all(np.abs(got - X64 @ W64[:m].T) <= bound[:, :m]), (rep, m)
        hip.hipGraphExecDestroy(exe)
        hip.hipGraphDestroy(graph)


@pytest.mark.gpu
@pytest.mark.parametrize("N,K", [(3, 96), (70, 2592), (2, 70016)])
def test_unaligned_activations(N, K):
    """X that is only 4-byte aligned (a slice of a caller's buffer): the split
    into planes falls back to 4-byte loads."""
    rng = np.random.default_rng(N + K)
    W = ((rng.standard_normal((64, K)) / 64).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    X = rng.standard_normal((N, K)).astype(np.float32)
    with G.Context(G.default_config(max_context=256, num_layers=6), 256) as ctx:
        dW, dC = DeviceBuffer.of(W), DeviceBuffer(N * 64 * 4)
        dX = DeviceBuffer.of(np.concatenate([np.zeros(1, np.float32), X.reshape(-1)]))
        ctx.matmul_bf16_device(dC.ptr, dW.ptr, dX.ptr + 4, N, 64, K)
        got = dC.download(np.float32, (N, 64)).astype(np.float64)
    W64, X64 = (W.astype(np.uint32) << 16).view(np.float32).astype(np.float64), X.astype(np.float64)
    bound = (2.0 ** -16 + K * 2.0 ** -24) * (np.abs(X64) @ np.abs(W64).T)
    assert np.all(np.abs(got - X64 @ W64.T) <= bound)


@pytest.mark.gpu
@pytest.mark.parametrize("hidden", [32, 1056, 2080, 3104, 8192])
def test_row_lengths(hidden):
    """The per-row norm and residual steps at each row length class (1, 2, 3,
    4 and 8 groups of four values per thread): a one-layer batched prefill
    against the token forward over the same tokens, at the 1e-3 x RMS bar of
    the whole-model test (x as two bf16 planes against fp32)."""
    batched_against_token_loop(17, hidden, 64)


@pytest.mark.gpu
@pytest.mark.parametrize("n,hidden", [(16, 32), (64, 96), (65, 64), (96, 1056), (97, 2080), (128, 96)])
def test_gate_up_token_classes(n, hidden):
    """Gate and up as a weight stream at the edges of its token classes (32,
    64, 96 and 128 per workgroup), one to three chunks of K per split."""
    batched_against_token_loop(n, hidden, 288)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [32, 64, 96, 128])
def test_gate_up_rings_turn_over(n):
    """The same classes at Gemma3-4B's sizes, where a split walks 13 or 14
    chunks through rings of two and three slots: the counted waits in their
    steady state, against the token forward."""
    kind, splits = plan(n, 2560, [10240, 10240], 1)
    assert kind == WIDE and 40 // splits >= 8
    batched_against_token_loop(n, 2560, 10240)


def random_model(rng, hidden, inter, vocab, layers):
    """Host weights of a small model at the default 8 / 4 heads of 256."""
    def w(*shape, scale):
        return ((rng.standard_normal(shape) * scale).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)

    s = 1 / np.sqrt(hidden)
    layers = [dict(input_layernorm=w(hidden, scale=0.1), q_proj=w(2048, hidden, scale=s), k_proj=w(1024, hidden, scale=s),
                   v_proj=w(1024, hidden, scale=s), o_proj=w(hidden, 2048, scale=0.02), q_norm=w(256, scale=0.1),
                   k_norm=w(256, scale=0.1), post_attention_layernorm=w(hidden, scale=0.1),
                   gate_proj=w(inter, hidden, scale=s), up_proj=w(inter, hidden, scale=s),
                   down_proj=w(hidden, inter, scale=0.1), pre_feedforward_layernorm=w(hidden, scale=0.1),
                   post_feedforward_layernorm=w(hidden, scale=0.1)) for _ in range(layers)]
    return G.host_weights(w(vocab, hidden, scale=1.0), layers, w(hidden, scale=0.1))


def batched_against_token_loop(n, hidden, inter):
    vocab = 96
    rng = np.random.default_rng(hidden)
    HW, keep = random_model(rng, hidden, inter, vocab, 1)
    tokens = rng.integers(0, vocab, n).astype(np.int32)
    cfg = G.default_config(num_layers=1, hidden_size=hidden, intermediate_size=inter, vocab_size=vocab, max_context=max(64, n))
    with G.Context(cfg, max(64, n)) as ctx:
        ctx.upload_weights(HW)
        got = ctx.prefill_tokens(tokens)
        for i, t in enumerate(tokens):
            want = ctx.forward_token(t, i)
    e = float(np.max(np.abs(got - want)) / np.sqrt(np.mean(want.astype(np.float64) ** 2)))
    print(f"[rows n={n} hidden={hidden}] batched vs token loop {e:.2e}", flush=True)
    assert e <= 1e-3
