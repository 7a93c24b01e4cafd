"""nf_hip_run_tasks merges adjacent decode GEMVs and small-batch linears
that read the same activation buffer (q/k/v, gate/up) into one launch, and
pairs of layer ops (two ropes, add and norm, silu and product).  Each
result must be bit-identical to dispatching the tasks one by one, the launch
count must show the merge, and a hazard between two tasks (here: both write
the same output; a weight buffer written mid-list; each task reading the
previous one's output) must keep the order."""
import ctypes as C

import numpy as np
import pytest

from helpers import assert_close
from neurofabric_amd import abi
from neurofabric_amd import synthetic as syn
from neurofabric_amd.abi import nf_task_desc

pytestmark = pytest.mark.gpu

QDT = {"q4_0": abi.NF_DTYPE_Q4_0, "q8_0": abi.NF_DTYPE_Q8_0}


def _array(tasks):
    arr = (nf_task_desc * len(tasks))()
    for i, td in enumerate(tasks):
        C.memmove(C.addressof(arr[i]), C.addressof(td), C.sizeof(nf_task_desc))
        arr[i].user_data = C.addressof(arr[i])
    return arr


def _block(provider, fmt, f16, M, hidden, kv, ffn, seed):
    """One Llama block's projections with the model's dataflow."""
    adt = abi.NF_DTYPE_F16 if f16 else abi.NF_DTYPE_F32
    npdt = np.float16 if f16 else np.float32
    elt = 2 if f16 else 4
    acts = {r: provider.alloc_array(syn.activations(M, k, seed=seed + i, dtype=npdt), adt)
            for i, (r, k) in enumerate((("attn_norm", hidden), ("attn_out", hidden), ("ffn_norm", hidden),
                                       ("ffn_act", ffn)))}
    projs = [("q", "attn_norm", hidden, hidden), ("k", "attn_norm", kv, hidden), ("v", "attn_norm", kv, hidden),
             ("o", "attn_out", hidden, hidden), ("gate", "ffn_norm", ffn, hidden), ("up", "ffn_norm", ffn, hidden),
             ("down", "ffn_act", hidden, ffn)]
    host_w, bufs, outs, specs = {}, [], {}, []
    op = f"dequant_{fmt}_linear" + ("_f16" if f16 else "")
    for j, (name, role, N, K) in enumerate(projs):
        host_w[name] = syn.weights(fmt, N, K, seed=seed + 10 + j)
        w = provider.alloc_array(host_w[name], QDT[fmt])
        outs[name] = provider.alloc(adt, M * N * elt)
        bufs.append(w)
        specs.append((name, role, w, N, K))
    tasks = [provider.task(op, [acts[role], w], [outs[name]], M, N, K) for (name, role, w, N, K) in specs]
    return op, acts, outs, specs, tasks, bufs + list(acts.values()) + list(outs.values()), host_w


@pytest.mark.parametrize("fmt", ["q4_0", "q8_0"])
@pytest.mark.parametrize("f16", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("M", [1, 3, 8, 16])
def test_run_tasks_merges_same_input_gemvs(provider, oracle_mod, fmt, f16, M):
    """M <= 4: decode GEMV groups; M = 8, 16: small-batch MFMA groups."""
    hidden, kv, ffn = 1024, 128, 2816
    op, acts, outs, specs, tasks, bufs, host_w = _block(provider, fmt, f16, M, hidden, kv, ffn, seed=M * 7)
    npdt = np.float16 if f16 else np.float32
    try:
        arr = _array(tasks)
        before = provider.launch_count()
        provider.run_tasks(arr, 1)
        provider.synchronize()
        assert provider.launch_count() - before == 4  # q+k+v, o, gate+up, down
        grouped = {name: outs[name].download(npdt).copy() for (name, *_r) in specs}
        # the same tasks one dispatch each
        for (name, role, w, N, K) in specs:
            provider.dispatch(op, [acts[role], w], [outs[name]], M, N, K)
        provider.synchronize()
        for (name, *_r) in specs:
            single = outs[name].download(npdt)
            assert np.array_equal(grouped[name].view(np.uint8), single.view(np.uint8)), name
        # and one merged member against the oracle
        A = acts["attn_norm"].download(npdt).reshape(M, hidden)
        ref = oracle_mod.fused(A, host_w["k"], fmt, M, kv, hidden, f16=f16, threads=8)
        if f16:
            ref = ref.view(np.float16)
        assert_close(grouped["k"].reshape(M, kv).astype(np.float32), ref.astype(np.float32), what=f"{fmt} k")
    finally:
        for b in bufs:
            b.release()


def _merged_and_apart(provider, fmt, f16, M, Ns, K, seed=0):
    """Linears of `Ns` weight rows over one activation buffer, as a list and
    then one dispatch each: (launches of the list, outputs equal bit for
    bit, the inputs, weights and outputs)."""
    npdt, dt = (np.float16, abi.NF_DTYPE_F16) if f16 else (np.float32, abi.NF_DTYPE_F32)
    op = f"dequant_{fmt}_linear" + ("_f16" if f16 else "")
    A = syn.activations(M, K, seed=seed + M, dtype=npdt)
    Ws = [syn.weights(fmt, N, K, seed=seed + i) for i, N in enumerate(Ns)]
    a = provider.alloc_array(A, dt)
    ws = [provider.alloc_array(W, QDT[fmt]) for W in Ws]
    cs = [provider.alloc(dt, M * N * A.itemsize) for N in Ns]
    try:
        arr = _array([provider.task(op, [a, w], [c], M, N, K) for w, c, N in zip(ws, cs, Ns)])
        before = provider.launch_count()
        provider.run_tasks(arr, 2)  # twice: the split-K counters must be back at zero
        provider.synchronize()
        launches = provider.launch_count() - before
        assert launches % 2 == 0
        merged = [c.download(npdt).copy() for c in cs]
        for w, c, N in zip(ws, cs, Ns):
            provider.dispatch(op, [a, w], [c], M, N, K)
        provider.synchronize()
        single = [c.download(npdt).copy() for c in cs]
    finally:
        for b in [a] + ws + cs:
            b.release()
    equal = [np.array_equal(x.view(np.uint8), y.view(np.uint8)) for x, y in zip(merged, single)]
    return launches // 2, equal, A, Ws, [x.reshape(M, N) for x, N in zip(merged, Ns)]


@pytest.mark.parametrize("fmt", ["q4_0", "q8_0"])
@pytest.mark.parametrize("M", [24, 48, 100])
@pytest.mark.parametrize("Ns,K", [((640, 640, 640), 1024), ((2048, 256, 256), 2048), ((1500, 1500), 768)],
                         ids=["qkv", "gqa", "gate_up"])
def test_run_tasks_merges_f16_batches(provider, oracle_mod, fmt, M, Ns, K):
    """f16 batches past 16 rows are small-batch launches by default, so lists
    merge them too; every output has the bits of its own dispatch.  Equal
    linears always share a launch (one variant and K split)."""
    launches, equal, A, Ws, out = _merged_and_apart(provider, fmt, True, M, Ns, K, seed=K)
    assert all(equal), equal
    assert launches == 1 if len(set(Ns)) == 1 else launches <= len(Ns)
    for W, N, c in zip(Ws, Ns, out):
        ref = oracle_mod.fused(A, W, fmt, M, N, K, f16=True, threads=8).view(np.float16)
        assert_close(c.astype(np.float32), ref.astype(np.float32), what=f"{fmt} {M}x{N}x{K}")


@pytest.mark.parametrize("fmt", ["q4_0", "q8_0"])
@pytest.mark.parametrize("M", [24, 33, 64])
@pytest.mark.parametrize("Ns,K", [((1024, 128, 128), 1024), ((2816, 2816), 1024), ((33, 700, 257, 1), 768)],
                         ids=["gqa", "gate_up", "ragged"])
def test_run_tasks_merges_f32_batches(provider, oracle_mod, fmt, M, Ns, K):
    """f32 batches of two and four activation tiles off the ring kernel: one
    launch, each linear with the K split, and the bits, of its own."""
    launches, equal, A, Ws, out = _merged_and_apart(provider, fmt, False, M, Ns, K, seed=K)
    assert all(equal), equal
    assert launches == 1
    for W, N, c in zip(Ws, Ns, out):
        assert_close(c, oracle_mod.fused(A, W, fmt, M, N, K, threads=8), what=f"{fmt} {M}x{N}x{K}")


# (format, f16, M, weight rows, K, launches): linears whose K splits add up to
# more than one round of workgroups, one launch all the same; weights of more
# than 16384 rows, whose sums run in another order, or of the f32 ring kernel
# (Q4_0 above 8192 rows at M = 33..64), first in the list: alone, the rest
# merged.
@pytest.mark.parametrize("fmt,f16,M,Ns,K,launches", [
    ("q4_0", False, 24, (8192, 1024, 1024), 8192, 1),
    ("q8_0", False, 64, (2048, 300, 1100), 2048, 1),
    ("q8_0", False, 40, (5632, 5632), 2048, 1),
    ("q8_0", False, 64, (1024, 256, 256), 4096, 1),
    ("q4_0", False, 24, (16400, 512, 640), 256, 2),
    ("q8_0", False, 24, (16400, 512, 640), 256, 2),
    ("q4_0", False, 48, (8200, 512, 640), 512, 2),
    ("q4_0", False, 48, (8200, 16000), 512, 1),
    ("q4_0", True, 12, (8192, 1024, 1024), 8192, 1),
], ids=lambda v: str(v))
def test_run_tasks_merges_uneven_linears(provider, fmt, f16, M, Ns, K, launches):
    got, equal, _, _, out = _merged_and_apart(provider, fmt, f16, M, Ns, K, seed=M)
    assert all(equal), equal
    assert got == launches
    assert all(np.isfinite(x).all() for x in out)


def test_run_tasks_keeps_hazards_apart(provider, oracle_mod):
    """Two GEMVs over the same activations that write the same output are
    not merged; the output is the second one's, as in dispatch order."""
    M, N, K = 1, 300, 512
    A = syn.activations(M, K, seed=1)
    W1, W2 = syn.q4_0_weights(N, K, seed=2), syn.q4_0_weights(N, K, seed=3)
    a = provider.alloc_array(A, abi.NF_DTYPE_F32)
    w1 = provider.alloc_array(W1, abi.NF_DTYPE_Q4_0)
    w2 = provider.alloc_array(W2, abi.NF_DTYPE_Q4_0)
    c = provider.alloc(abi.NF_DTYPE_F32, M * N * 4)
    try:
        arr = _array([provider.task("dequant_q4_0_linear", [a, w], [c], M, N, K) for w in (w1, w2)])
        before = provider.launch_count()
        provider.run_tasks(arr, 1)
        provider.synchronize()
        assert provider.launch_count() - before == 2
        assert_close(c.download(np.float32).reshape(M, N), oracle_mod.fused(A, W2, "q4_0", M, N, K))
    finally:
        for b in (a, w1, w2, c):
            b.release()


def test_run_tasks_weight_written_mid_list(provider, oracle_mod):
    """A task in the middle of a batch overwrites the weight buffer a later
    GEMV reads (embedding_lookup copying new Q4_0 bytes into it, bit for
    bit); the later GEMV must use the new bytes, also when the list is run
    twice in one call (repeat=2)."""
    from neurofabric_amd.plugin import push_constants
    M, N, K = 1, 300, 512
    A = syn.activations(M, K, seed=5)
    W1, W2_old, W2_new = (syn.q4_0_weights(N, K, seed=s) for s in (6, 7, 8))
    assert W2_new.nbytes % 4 == 0
    dim = W2_new.nbytes // 4
    a = provider.alloc_array(A, abi.NF_DTYPE_F32)
    w1 = provider.alloc_array(W1, abi.NF_DTYPE_Q4_0)
    w2 = provider.alloc_array(W2_old.view(np.float32), abi.NF_DTYPE_F32)
    table = provider.alloc_array(W2_new.view(np.float32), abi.NF_DTYPE_F32)
    ids = provider.alloc_array(np.zeros(1, np.int32), abi.NF_DTYPE_I32)
    c1 = provider.alloc(abi.NF_DTYPE_F32, M * N * 4)
    c2 = provider.alloc(abi.NF_DTYPE_F32, M * N * 4)
    try:
        arr = _array([provider.task("dequant_q4_0_linear", [a, w1], [c1], M, N, K),
                      provider.task("embedding_lookup", [table, ids], [w2], pc=push_constants(seq_len=1, head_dim=dim)),
                      provider.task("dequant_q4_0_linear", [a, w2], [c2], M, N, K)])
        provider.run_tasks(arr, 2)
        provider.synchronize()
        assert np.array_equal(w2.download(np.uint8), W2_new)
        assert_close(c1.download(np.float32).reshape(M, N), oracle_mod.fused(A, W1, "q4_0", M, N, K), what="first")
        assert_close(c2.download(np.float32).reshape(M, N), oracle_mod.fused(A, W2_new, "q4_0", M, N, K),
                     what="after the write")
    finally:
        for b in (a, w1, w2, table, ids, c1, c2):
            b.release()


@pytest.mark.parametrize("fmt", ["q4_0", "q8_0"])
def test_run_tasks_chain_bit_identical(provider, fmt):
    """Twelve decode GEMVs with distinct weights and shapes, the adjacent
    same-input ones merged, through nf_hip_run_tasks three times in one
    call, then one dispatch each: bit-identical outputs."""
    M, K = 1, 2048
    A = syn.activations(M, K, seed=9)
    a = provider.alloc_array(A, abi.NF_DTYPE_F32)
    shapes = [2048, 256, 256, 2048, 5632, 5632, 2048, 1024, 4096, 300, 64, 8192]
    bufs, tasks, outs = [a], [], []
    op = f"dequant_{fmt}_linear"
    for i, N in enumerate(shapes):
        w = provider.alloc_array(syn.weights(fmt, N, K, seed=20 + i), QDT[fmt])
        c = provider.alloc(abi.NF_DTYPE_F32, M * N * 4)
        bufs += [w, c]
        outs.append((w, c, N))
        tasks.append(provider.task(op, [a, w], [c], M, N, K))
    try:
        provider.run_tasks(_array(tasks), 3)
        provider.synchronize()
        got = [c.download(np.float32).copy() for (_, c, _) in outs]
        for (w, c, N) in outs:
            provider.dispatch(op, [a, w], [c], M, N, K)
        provider.synchronize()
        for i, (_, c, _) in enumerate(outs):
            assert np.array_equal(got[i].view(np.uint32), c.download(np.float32).view(np.uint32)), i
    finally:
        for b in bufs:
            b.release()


@pytest.mark.parametrize("fmt", ["q4_0", "q8_0"])
@pytest.mark.parametrize("f16", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("dims", [(2048, 1024, 64, 5632, 2048, 128, 4096), (512, 256, 64, 256, 1024)],
                         ids=["mixed", "small"])
def test_run_tasks_dependent_sequence(provider, oracle_mod, fmt, f16, dims):
    """Decode GEMVs where each reads the previous one's output (layer i:
    K = dims[i], N = dims[i+1]), some with few rows: one launch each (no
    two share an input), bit-identical to one dispatch each, in order; the
    first layer against the oracle."""
    M = 1
    adt = abi.NF_DTYPE_F16 if f16 else abi.NF_DTYPE_F32
    npdt = np.float16 if f16 else np.float32
    op = f"dequant_{fmt}_linear" + ("_f16" if f16 else "")
    x0 = syn.activations(M, dims[0], seed=31, dtype=npdt)
    acts = [provider.alloc_array(x0, adt)] + [provider.alloc(adt, M * n * x0.itemsize) for n in dims[1:]]
    host_w, ws, tasks = [], [], []
    for i in range(len(dims) - 1):
        K, N = dims[i], dims[i + 1]
        host_w.append(syn.weights(fmt, N, K, seed=40 + i))
        ws.append(provider.alloc_array(host_w[-1], QDT[fmt]))
        tasks.append(provider.task(op, [acts[i], ws[-1]], [acts[i + 1]], M, N, K))
    try:
        before = provider.launch_count()
        provider.run_tasks(_array(tasks), 1)
        provider.synchronize()
        assert provider.launch_count() - before == len(tasks)
        chained = [a.download(npdt).copy() for a in acts[1:]]
        for t_i in range(len(tasks)):
            K, N = dims[t_i], dims[t_i + 1]
            provider.dispatch(op, [acts[t_i], ws[t_i]], [acts[t_i + 1]], M, N, K)
        provider.synchronize()
        for i, a in enumerate(acts[1:]):
            assert np.array_equal(chained[i].view(np.uint8), a.download(npdt).view(np.uint8)), f"layer {i}"
        ref = oracle_mod.fused(x0, host_w[0], fmt, M, dims[1], dims[0], f16=f16, threads=8)
        if f16:
            ref = ref.view(np.float16)
        assert_close(chained[0].reshape(M, dims[1]).astype(np.float32), ref.astype(np.float32), what=f"{fmt} layer 0")
    finally:
        for b in acts + ws:
            b.release()


# A layer op and the one after it in one launch: per pair, the ops as (op,
# inputs, output) over named buffers, and the launches expected for rows of a
# whole number of 16-byte chunks.  "a", "b" and "u" hold data, "w" f32 weights.
FUSED = {
    "rope": ([("rope_batch", ["a"], "s"), ("rope_batch", ["b"], "t")], 1),
    "rope_in_place": ([("rope_batch", ["a"], "a"), ("rope_batch", ["b"], "b")], 1),
    "rope_chained": ([("rope_batch", ["a"], "s"), ("rope_batch", ["s"], "t")], 2),
    "rope_silu": ([("rope_batch", ["a"], "s"), ("silu", ["b"], "t")], 2),
    "add_norm": ([("metal_vector_add", ["a", "b"], "s"), ("rms_norm", ["s", "w"], "t")], 1),
    "add_norm_residual": ([("metal_vector_add", ["a", "b"], "a"), ("rms_norm", ["a", "w"], "t")], 1),
    "add_norm_overwrites": ([("metal_vector_add", ["a", "b"], "s"), ("rms_norm", ["s", "w"], "b")], 2),
    "add_norm_in_place": ([("metal_vector_add", ["a", "b"], "s"), ("rms_norm", ["s", "w"], "s")], 2),
    "silu_mul": ([("silu", ["a"], "s"), ("elementwise_mul", ["s", "u"], "t")], 1),
    "silu_mul_swapped": ([("silu", ["a"], "s"), ("elementwise_mul", ["u", "s"], "t")], 1),
    "silu_mul_in_place": ([("silu", ["a"], "a"), ("elementwise_mul", ["a", "u"], "u")], 1),
    "silu_mul_onto_gate": ([("silu", ["a"], "s"), ("elementwise_mul", ["s", "u"], "a")], 1),
    "silu_squared": ([("silu", ["a"], "s"), ("elementwise_mul", ["s", "s"], "t")], 2),
    "silu_add": ([("silu", ["a"], "s"), ("metal_vector_add", ["s", "u"], "t")], 2),
}


@pytest.mark.parametrize("f16", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("rows,dim", [(1, 64), (3, 2048), (2, 260), (5, 30), (1, 8192), (600, 128)],
                         ids=lambda v: str(v))
@pytest.mark.parametrize("pair", sorted(FUSED))
def test_run_tasks_layer_pairs(provider, pair, rows, dim, f16):
    """Both outputs bit-identical to one dispatch each, with infinities and
    NaN among the inputs; rows that are no whole number of 16-byte chunks
    (260 halves, 30 elements) and operands in the way take two launches.
    The second rope has fewer heads than the first."""
    from neurofabric_amd.plugin import push_constants
    npdt, dt = (np.float16, abi.NF_DTYPE_F16) if f16 else (np.float32, abi.NF_DTYPE_F32)
    rng = np.random.default_rng(rows * dim + f16)
    data = {n: rng.standard_normal((rows, dim)).astype(npdt) for n in "abust"}
    data["a"][0, :3] = np.inf, -np.inf, np.nan
    data["u"][-1, -1] = -np.inf
    data["w"] = rng.standard_normal(dim).astype(np.float32)
    bufs = {n: provider.alloc_array(x, abi.NF_DTYPE_F32 if n == "w" else dt) for n, x in data.items()}
    steps, launches = FUSED[pair]
    heads = 2 if rows % 2 == 0 else 1
    tasks = [provider.task(op, [bufs[n] for n in ins], [bufs[out]],
                           pc=push_constants(seq_len=rows, n_heads=heads if i == 0 else 1, head_dim=dim, epsilon=1e-5,
                                             theta=10000.0, step_idx=7))
             for i, (op, ins, out) in enumerate(steps)]
    if not pair.startswith("rope"):
        per = 8 if f16 else 4
        # the norm needs whole chunks of a row, silu and mul only aligned buffers
        if pair.startswith("add") and dim % per:
            launches = 2
    try:
        before = provider.launch_count()
        provider.run_tasks(_array(tasks), 1)
        provider.synchronize()
        assert provider.launch_count() - before == launches
        got = {n: b.download(data[n].dtype).copy() for n, b in bufs.items()}
        for n, b in bufs.items():
            b.upload(data[n])
        for td in tasks:
            provider.check(provider.dispatch_task(td), "dispatch")
        provider.synchronize()
        for n, b in bufs.items():
            assert np.array_equal(got[n].view(np.uint8), b.download(data[n].dtype).view(np.uint8)), n
    finally:
        for b in bufs.values():
            b.release()


@pytest.mark.parametrize("f16", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("tok,heads,D", [(1, (32, 8), 64), (5, (4, 12), 96), (130, (7, 1), 128), (700, (8, 2), 64)],
                         ids=lambda v: str(v))
def test_run_tasks_rope_pair_of_two_sizes(provider, tok, heads, D, f16):
    """q and k of different head counts, the larger first or second, one
    launch: the second job's workgroups begin where the first's end, and each
    has its own group size.  The bits of one dispatch each."""
    from neurofabric_amd.plugin import push_constants
    npdt, dt = (np.float16, abi.NF_DTYPE_F16) if f16 else (np.float32, abi.NF_DTYPE_F32)
    rng = np.random.default_rng(tok + D)
    xs = [rng.standard_normal(tok * h * D).astype(npdt) for h in heads]
    ins = [provider.alloc_array(x, dt) for x in xs]
    outs = [provider.alloc(dt, x.nbytes) for x in xs]
    tasks = [provider.task("rope_batch", [a], [o], pc=push_constants(seq_len=tok, n_heads=h, head_dim=D, theta=1e4,
                                                                     step_idx=11)) for a, o, h in zip(ins, outs, heads)]
    try:
        before = provider.launch_count()
        provider.run_tasks(_array(tasks), 1)
        provider.synchronize()
        assert provider.launch_count() - before == 1
        got = [o.download(npdt).copy() for o in outs]
        for td in tasks:
            provider.check(provider.dispatch_task(td), "dispatch")
        provider.synchronize()
        for g, o in zip(got, outs):
            assert np.array_equal(g.view(np.uint8), o.download(npdt).view(np.uint8))
    finally:
        for b in ins + outs:
            b.release()


# Two NaNs of different payloads meet in the product and in the sum: the bits
# of the fused launches are those of the separate ones for either operand order.
@pytest.mark.parametrize("f16", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("pair,dim", [("add_norm", 64), ("silu_mul", 64), ("silu_mul", 30), ("silu_mul_swapped", 64),
                                      ("silu_mul_swapped", 30)])
def test_run_tasks_layer_pairs_nan_payloads(provider, pair, dim, f16):
    from neurofabric_amd.plugin import push_constants
    npdt, ut, dt = (np.float16, np.uint16, abi.NF_DTYPE_F16) if f16 else (np.float32, np.uint32, abi.NF_DTYPE_F32)
    one = 0x7E01 if f16 else 0x7FC00001
    data = {n: np.ones((3, dim), npdt) for n in "abust"}
    for i, n in enumerate("abu"):
        data[n].view(ut)[...] = one + np.arange(3 * dim, dtype=ut).reshape(3, dim) % 50 + 64 * i
    for n in "bu":
        data[n].view(ut)[1] |= 0x8000 if f16 else 0x80000000
    data["w"] = np.ones(dim, np.float32)
    bufs = {n: provider.alloc_array(x, abi.NF_DTYPE_F32 if n == "w" else dt) for n, x in data.items()}
    steps, launches = FUSED[pair]
    tasks = [provider.task(op, [bufs[n] for n in ins], [bufs[out]],
                           pc=push_constants(seq_len=3, n_heads=1, head_dim=dim, epsilon=1e-5))
             for op, ins, out in steps]
    try:
        before = provider.launch_count()
        provider.run_tasks(_array(tasks), 1)
        provider.synchronize()
        assert provider.launch_count() - before == launches
        got = {n: b.download(data[n].dtype).copy() for n, b in bufs.items()}
        for td in tasks:
            provider.check(provider.dispatch_task(td), "dispatch")
        provider.synchronize()
        for n, b in bufs.items():
            assert np.array_equal(got[n].view(np.uint8), b.download(data[n].dtype).view(np.uint8)), n
    finally:
        for b in bufs.values():
            b.release()
