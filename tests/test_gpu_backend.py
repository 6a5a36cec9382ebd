"""The plugin impl's forward on the GPU against the oracle's restatement of the
reference backend (backend.py:249-393): writes, window tags, and attention routed to
fresh-only prefill, split-K decode / MTP and continuation prefill, in bf16 and fp16."""
import numpy as np
import pytest
import torch

from oracle import backend as ob
from oracle import cases

pytestmark = pytest.mark.gpu


class _Layer:
    layer_name = "model.layers.3.self_attn.attn"


class _MD:
    pass


@pytest.mark.parametrize("qdt,ulp", [(torch.bfloat16, 2.0 ** -7), (torch.float16, 2.0 ** -10)],
                         ids=["bf16", "fp16"])
def test_forward_steps_match_oracle(cuda, qdt, ulp):
    from oscar_amd.backend import OscarAttentionBackendImpl

    dev = torch.device("cuda", 0)
    d, hq, hk, bs = 256, 6, 1, 128
    impl = OscarAttentionBackendImpl.__new__(OscarAttentionBackendImpl)
    impl.head_size, impl.num_heads, impl.num_kv_heads, impl.scale = d, hq, hk, d ** -0.5
    impl.key_cache = impl.value_cache = None
    impl._oscar_setup()
    layer = _Layer()
    rk, rv = cases.hadamard_rotation(d, 5), cases.qr_rotation(d, 6)
    layer._oscar_rots = (torch.from_numpy(rk).to(dev), torch.from_numpy(rv).to(dev))
    nb, per = 24, 12
    caches = [torch.zeros(nb, bs, hk, d, dtype=torch.int8, device=dev) for _ in range(2)]
    table = np.random.default_rng(7).permutation(nb).reshape(2, per).astype(np.int32)
    oracle_layer = ob.OracleLayer(k8=np.zeros((nb, bs, hk, d), np.uint8), v8=np.zeros((nb, bs, hk, d), np.uint8),
                                  rk=rk, rv=rv, hq=hq, hk=hk, d=d, scale=d ** -0.5)
    q_dtype = "bf16" if qdt == torch.bfloat16 else "f16"
    lens = [0, 0]
    # (new tokens of request 0, of request 1): fresh prefills, MTP + single-token
    # decode, continuation chunks of 1200 and 2400 rows (the split-K decode, as 32-row
    # sub-requests) beside a decode and an MTP step (the continuation prefill through
    # the forward: test_config5_batched_forward)
    for step, (n0, n1) in enumerate([(300, 700), (4, 1), (200, 1), (400, 3)]):
        news = [n0, n1]
        slots, qsl, seqs = [], [0], []
        for r, n in enumerate(news):
            pos = np.arange(lens[r], lens[r] + n)
            slots += (table[r, pos // bs].astype(np.int64) * bs + pos % bs).tolist()
            qsl.append(qsl[-1] + n)
            seqs.append(lens[r] + n)
        N = qsl[-1]
        q = cases.bf16_normal((N, hq, d), 100 + step)
        k = cases.kv_outliers(N, hk, d, 200 + step)
        v = cases.kv_outliers(N, hk, d, 300 + step)
        md = _MD()
        md.num_actual_tokens = N
        md.slot_mapping = torch.tensor(slots, device=dev)
        md.query_start_loc_cpu = torch.tensor(qsl)
        md.seq_lens_list = seqs
        md.block_tables = torch.from_numpy(table).to(dev)
        out = torch.empty(N, hq * d, dtype=qdt, device=dev)
        tq, tk, tv = (torch.from_numpy(x).to(dev).to(qdt) for x in (q, k, v))
        impl.forward(layer, tq.view(N, -1), tk.view(N, -1), tv.view(N, -1), caches, md, output=out)
        torch.cuda.synchronize()
        ref = ob.forward(oracle_layer, q, k, v, slots, qsl, seqs, table, q_dtype=q_dtype)
        got = out.float().view(N, hq, d).cpu().numpy()
        # 2e-2 absolute plus one output ulp of the value (outlier channels make early
        # causal rows large, where one ulp exceeds 2e-2)
        excess = float((np.abs(got - ref) - (2e-2 + ulp * np.abs(ref))).max())
        print(f"{q_dtype} step {step}: max|out - oracle| = {np.abs(got - ref).max():.3e}", flush=True)
        assert excess <= 0, f"step {step}: output differs from the oracle"
        lens = seqs
    assert np.array_equal(layer._oscar_slot_owner.cpu().numpy(), oracle_layer.staging.owner)
    assert np.array_equal(caches[0].view(torch.uint8).cpu().numpy(), oracle_layer.k8)
    assert np.array_equal(caches[1].view(torch.uint8).cpu().numpy(), oracle_layer.v8)


@pytest.mark.parametrize("mode", ["mtp_window", "cache_only", "fp16_mtp", "long_chunks", "long_chunks_fresh",
                                  "fresh_last"])
def test_native_decode_step_matches_general_path_and_oracle(cuda, mode):
    """forward() on decode-shaped batches takes oscar_decode_step_v1 (one native call);
    the same batch through the general Python path (_run) and the oracle agree.
    long_chunks: chunks of 240 and 72 rows per KV head (sub-requests of the plan);
    long_chunks_fresh: the same beside a history-free request, which the native step
    declines and the general path routes as a compact decode batch (gathered rows and
    block-table rows, the fresh request lying between decodes) plus a prefill;
    fresh_last: the fresh request after the decodes (their rows and table rows are a
    slice of the batch's)."""
    from oscar_amd import backend as B
    from oracle.attention import attention_ref

    dev = torch.device("cuda", 0)
    qdt = torch.float16 if mode == "fp16_mtp" else torch.bfloat16
    fresh = mode != "cache_only"
    prefixes, lengths = [3000, 129, 700, 24579], [4, 1, 3, 4]
    if mode == "long_chunks":
        lengths = [40, 1, 12, 4]
    if mode == "long_chunks_fresh":
        prefixes, lengths = [3000, 0, 700, 24579], [40, 300, 12, 4]
    if mode == "fresh_last":
        prefixes, lengths = [3000, 700, 24579, 0], [40, 12, 4, 300]
    c = cases.make_case(prefixes, lengths, fresh=fresh, seed=77)
    d, hq, hk = 256, 6, 1
    impl = OscarAttentionBackendImplFactory()
    layer = _Layer()
    eye = torch.eye(d, dtype=torch.float32, device=dev)
    layer._oscar_rots = (eye, eye)
    caches = [torch.from_numpy(c[x]).view(torch.int8).to(dev) for x in ("k8", "v8")]
    impl._set_caches(caches)
    impl._ensure_staging(layer, caches)
    sk, sv, own = c["stage"]
    layer._oscar_stage_k.copy_(torch.from_numpy(sk))
    layer._oscar_stage_v.copy_(torch.from_numpy(sv))
    layer._oscar_slot_owner.copy_(torch.from_numpy(own))
    N = c["qsl"][-1]
    md = _MD()
    md.num_actual_tokens = N
    # the current chunk is not written (slots -1): the history and window stay the state
    md.slot_mapping = torch.full((N,), -1, dtype=torch.int64, device=dev)
    md.query_start_loc_cpu = torch.tensor(c["qsl"], dtype=torch.int32)
    md.seq_lens_cpu = torch.tensor(c["seqs"], dtype=torch.int32)
    md.block_tables = torch.from_numpy(c["bt"]).to(dev)
    tq = torch.from_numpy(c["q"]).to(dev).to(qdt).view(N, -1)
    tk = None if c["k"] is None else torch.from_numpy(c["k"]).to(dev).to(qdt).view(N, -1)
    tv = None if c["v"] is None else torch.from_numpy(c["v"]).to(dev).to(qdt).view(N, -1)
    calls = {"reads": impl._oscar_stats["reads"]}
    out_native = torch.empty(N, hq * d, dtype=qdt, device=dev)
    native = impl._native_step(layer, tq, tk, tv, caches, md, out_native)
    assert native == (mode not in ("long_chunks_fresh", "fresh_last"))
    out_general = torch.empty_like(out_native)
    impl._run(layer, tq, tk, tv, caches, md, out_general, write=True)
    torch.cuda.synchronize()
    assert impl._oscar_stats["reads"] == calls["reads"] + 1 + native
    if not native:
        out_native = out_general
    q_dtype = "f16" if qdt == torch.float16 else "bf16"
    ref_o, _ = attention_ref(c["q"], c["k"], c["v"], c["k8"], c["v8"], c["bt"], c["qsl"], c["seqs"],
                             c["scale"], c["stage"], q_dtype=q_dtype)
    ulp = 2.0 ** -7 if qdt == torch.bfloat16 else 2.0 ** -10
    for label, out in (("native", out_native), ("general", out_general)):
        got = out.float().view(N, hq, d).cpu().numpy()
        excess = float((np.abs(got - ref_o) - (2e-2 + ulp * np.abs(ref_o))).max())
        print(f"{mode} {label}: max|out - oracle| = {np.abs(got - ref_o).max():.3e}", flush=True)
        assert excess <= 0, f"{mode} {label} differs from the oracle"
    diff = (out_native.float() - out_general.float()).abs().max().item()
    print(f"{mode}: native vs general max diff {diff:.3e}", flush=True)
    assert diff <= 2e-2


@pytest.mark.parametrize("requests", [1, 21, 64, 65])
def test_native_step_metadata_follows_every_call(cuda, requests):
    """The step's plan and request table travel in the store's launch up to 64 tokens and in
    a copy of their own beyond.  Back to back steps whose lengths change from call to call
    (a stale or torn table shows) against the general path, bytes of the written slots
    included."""
    from oscar_amd.backend import OscarAttentionBackendImpl  # noqa: F401

    dev = torch.device("cuda", 0)
    d, hq, hk, bs = 256, 6, 1, 128
    g = np.random.default_rng(requests)
    prefixes = [int(x) for x in g.integers(40, 900, requests)]
    c = cases.make_case(prefixes, [1] * requests, seed=requests)
    table = torch.from_numpy(c["bt"]).to(dev)
    tq, tk, tv = (torch.from_numpy(c[x]).to(dev).bfloat16().view(requests, -1) for x in "qkv")
    results = []
    for native in (True, False):
        impl, layer = OscarAttentionBackendImplFactory(), _Layer()
        eye = torch.eye(d, dtype=torch.float32, device=dev)
        layer._oscar_rots = (eye, eye)
        caches = [torch.from_numpy(c[x]).view(torch.int8).to(dev).clone() for x in ("k8", "v8")]
        impl._set_caches(caches)
        impl._ensure_staging(layer, caches)
        for arena, x in zip((layer._oscar_stage_k, layer._oscar_stage_v, layer._oscar_slot_owner), c["stage"]):
            arena.copy_(torch.from_numpy(x))
        outs = []
        for step in range(6):
            lens = [p - step * (r % 3) for r, p in enumerate(prefixes)]  # read shorter histories
            md = _MD()
            md.num_actual_tokens = requests
            md.slot_mapping = torch.tensor([int(c["bt"][r, n // bs]) * bs + n % bs for r, n in enumerate(lens)], device=dev)
            md.query_start_loc_cpu = torch.arange(requests + 1, dtype=torch.int32)
            md.seq_lens_list = [n + 1 for n in lens]
            md.block_tables = table
            out = torch.empty(requests, hq * d, dtype=torch.bfloat16, device=dev)
            if native:
                assert impl._native_step(layer, tq, tk, tv, caches, md, out)
            else:
                impl._run(layer, tq, tk, tv, caches, md, out, write=True)
            outs.append(out)
        torch.cuda.synchronize()
        results.append((torch.stack(outs).float(), *caches, layer._oscar_slot_owner))
    (o1, k1, v1, w1), (o2, k2, v2, w2) = results
    assert torch.equal(k1, k2) and torch.equal(v1, v2) and torch.equal(w1, w2)
    # both paths round the output to bf16 once; sums may differ in order by one ulp of it
    excess = ((o1 - o2).abs() - (2e-3 + 2.0 ** -7 * o2.abs())).max().item()
    print(f"{requests} requests: native vs general past one ulp {excess:.2e}", flush=True)
    assert excess <= 0


# name: histories, chunks, and rows that belong to no request: before the first one, after
# the last one, past num_actual_tokens, and of the output alone
ROW_LAYOUTS = {
    "prompts": ([0, 0], [300, 41], 0, 0, 0, 0),
    "prompts, output of more rows": ([0, 0], [300, 41], 0, 0, 0, 9),
    "mixed, empty requests": ([700, 0, 300, 0, 129, 0], [3, 0, 0, 250, 1, 40], 0, 0, 0, 0),
    "mixed, output of more rows": ([700, 0], [3, 150], 0, 0, 0, 2),
    "mixed, padded query": ([700, 0], [3, 150], 0, 0, 7, 0),
    "mixed, rows before and after": ([0, 700], [150, 30], 3, 5, 0, 0),
    "prompt, rows after": ([0], [200], 0, 56, 0, 0),
    "decodes, rows after": ([700, 300], [1, 40], 0, 3, 2, 0),
    "decodes, rows before": ([700, 300], [1, 40], 2, 0, 0, 0),
}


@pytest.mark.parametrize("name", ROW_LAYOUTS)
def test_output_rows_are_written_or_zero(cuda, name):
    """The general path on an output full of NaN: a request's rows hold what the batch
    without any other rows gives, and every other row is zero."""
    prefixes, lengths, front, tail, pad, extra = ROW_LAYOUTS[name]
    dev = torch.device("cuda", 0)
    d, hq, hk = 256, 6, 1
    c = cases.make_case(prefixes, lengths, fresh=True, seed=41)
    used = c["qsl"][-1]
    eye = torch.eye(d, dtype=torch.float32, device=dev)

    def run(front, tail, pad, extra, fill):
        impl, layer = OscarAttentionBackendImplFactory(), _Layer()
        layer._oscar_rots = (eye, eye)
        caches = [torch.from_numpy(c[x]).view(torch.int8).to(dev).clone() for x in ("k8", "v8")]
        impl._set_caches(caches)
        impl._ensure_staging(layer, caches)
        for arena, x in zip((layer._oscar_stage_k, layer._oscar_stage_v, layer._oscar_slot_owner), c["stage"]):
            arena.copy_(torch.from_numpy(x))
        actual = front + used + tail
        md = _MD()
        md.num_actual_tokens = actual
        md.slot_mapping = torch.full((actual,), -1, dtype=torch.int64, device=dev)
        md.query_start_loc_cpu = torch.tensor([front + x for x in c["qsl"]], dtype=torch.int32)
        md.seq_lens_list = list(c["seqs"])
        md.block_tables = torch.from_numpy(c["bt"]).to(dev)
        rows = [torch.ones(actual + pad, h * d, dtype=torch.bfloat16, device=dev) for h in (hq, hk, hk)]
        for x, name in zip(rows, "qkv"):
            x[front:front + used] = torch.from_numpy(c[name]).to(dev).bfloat16().view(used, -1)
        out = torch.full((actual + pad + extra, hq * d), fill, dtype=torch.bfloat16, device=dev)
        impl._run(layer, *rows, caches, md, out, write=True)
        torch.cuda.synchronize()
        return out

    want = run(0, 0, 0, 0, 0.0)
    got = run(front, tail, pad, extra, float("nan"))
    assert torch.equal(got[front:front + used], want)
    assert (got[:front] == 0).all() and (got[front + used:] == 0).all()


def test_unread_long_requests_leave_zeros(cuda, monkeypatch):
    """More heads per KV head than a decode tile takes, without new tokens: nothing reads
    such a request, so its rows are zero (not the rotation of memory that nothing wrote)."""
    dev = torch.device("cuda", 0)
    d, hq = 256, 40
    c = cases.make_case([300, 500], [4, 60], group=hq, fresh=False, seed=43)
    impl, layer = OscarAttentionBackendImplFactory(), _Layer()
    impl.num_heads = hq
    eye = torch.eye(d, dtype=torch.float32, device=dev)
    layer._oscar_rots = (eye, eye)
    caches = [torch.from_numpy(c[x]).view(torch.int8).to(dev) for x in ("k8", "v8")]
    impl._set_caches(caches)
    md = _MD()
    md.num_actual_tokens = 64
    md.query_start_loc_cpu = torch.tensor(c["qsl"], dtype=torch.int32)
    md.seq_lens_list = list(c["seqs"])
    md.block_tables = torch.from_numpy(c["bt"]).to(dev)
    out = torch.full((64, hq * d), float("nan"), dtype=torch.bfloat16, device=dev)
    empty = torch.empty

    def holding_nan(*shape, **kw):
        x = empty(*shape, **kw)
        return x.fill_(float("nan")) if x.is_floating_point() else x

    monkeypatch.setattr(torch, "empty", holding_nan)
    impl._streaming_attention(layer, torch.from_numpy(c["q"]).to(dev).bfloat16().view(64, -1), None, None, caches, md, out)
    torch.cuda.synchronize()
    assert (out == 0).all()


def OscarAttentionBackendImplFactory():
    from oscar_amd.backend import OscarAttentionBackendImpl

    impl = OscarAttentionBackendImpl.__new__(OscarAttentionBackendImpl)
    impl.head_size, impl.num_heads, impl.num_kv_heads, impl.scale = 256, 6, 1, 256 ** -0.5
    impl.key_cache = impl.value_cache = None
    impl._oscar_setup()
    return impl
