"""Model-level GPU tests: prefill/decode consistency, engine batching
invariance, encoder contract."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tiny():
    from quickstart_streaming_agents_amd.models.llama import (LlamaConfig,
                                                              LlamaModel)
    return LlamaModel(LlamaConfig.preset("tiny"), device="cuda:0", seed=3)


def test_prefill_decode_consistency(tiny):
    """prefill(t)[last] must match prefill(t-1) -> decode(token t): the two
    paths (GEMM+softmax kernel vs paged-attention kernel) are numerically
    the same computation."""
    from quickstart_streaming_agents_amd.models.kv_cache import PagedKVCache
    torch.manual_seed(0)
    prompt = torch.randint(16, 2000, (75,), dtype=torch.int64, device="cuda:0")

    kv_a = tiny.new_kv_cache(16)
    kv_a.allocate(0, 75)
    logits_a = tiny.forward_prefill(prompt, kv_a, 0)

    kv_b = tiny.new_kv_cache(16)
    kv_b.allocate(0, 74)
    tiny.forward_prefill(prompt[:74], kv_b, 0)
    kv_b.extend(0, 75)
    bt = kv_b.block_table([0])
    sl = kv_b.seq_lens_tensor([0])
    pos = torch.tensor([74], dtype=torch.int32, device="cuda:0")
    logits_b = tiny.forward_decode(prompt[74:75], kv_b, bt, sl, pos)[0]

    torch.testing.assert_close(logits_a, logits_b, atol=8e-2, rtol=8e-2)
    assert int(logits_a.argmax()) == int(logits_b.argmax())


@pytest.mark.parametrize("rows", [1, 5, 33])
def test_decode_takes_tokens_as_the_embedding_does(tiny, rows):
    """i32 tokens and a strided column of them, on the fp8 streams and beyond
    their 32 rows."""
    assert tiny._streams_fp8()
    g = torch.Generator().manual_seed(rows)
    table = torch.randint(16, 2000, (rows, 3), generator=g).to("cuda:0")

    def step(tokens):
        kv = tiny.new_kv_cache(rows)
        for i in range(rows):
            kv.allocate(i, 1)
        ids = list(range(rows))
        lens = kv.seq_lens_tensor(ids)
        return tiny.forward_decode(tokens, kv, kv.block_table(ids), lens,
                                   lens - 1)

    want = step(table[:, 1].contiguous())
    assert torch.equal(step(table[:, 1]), want)
    assert torch.equal(step(table[:, 1].int()), want)
    assert torch.equal(step(table.int()[:, 1]), want)


def test_engine_determinism_and_shapes(tiny):
    """Greedy decode is deterministic across engines; output lengths honor
    max_new_tokens.  (Exact solo-vs-batched token equality is NOT asserted:
    with random-init weights logits are near-tied and bf16 GEMM shape
    differences legitimately flip argmax.)"""
    from quickstart_streaming_agents_amd.models.serve import Engine
    prompts = [[1, 5, 9, 200, 17], [1, 77, 31], [1, 5, 9, 200, 17, 40, 41]]
    e2 = Engine(tiny, max_batch=8, max_seq_len=256)
    batched = e2.generate_batch(prompts, [10, 10, 10])
    assert all(len(o) == 10 for o in batched)
    assert all(0 <= t < tiny.cfg.vocab_size for o in batched for t in o)
    # determinism across engines
    e3 = Engine(tiny, max_batch=8, max_seq_len=256)
    assert e3.generate_batch(prompts, [10, 10, 10]) == batched
    # graph path vs eager path agree on the FIRST decode token per seq
    # (same GEMM shapes at the first step after identical prefill)
    e4 = Engine(tiny, max_batch=8, max_seq_len=256)
    e4.use_graph = False
    eager = e4.generate_batch(prompts, [10, 10, 10])
    assert [o[0] for o in eager] == [o[0] for o in batched]


def test_engine_continuous_admission(tiny):
    """More sequences than max_batch complete correctly via admission."""
    from quickstart_streaming_agents_amd.models.serve import Engine
    e = Engine(tiny, max_batch=4, max_seq_len=128, kv_pages=20)
    prompts = [[1, i + 10, i + 20] for i in range(12)]
    outs = e.generate_batch(prompts, [6] * 12)
    assert len(outs) == 12 and all(len(o) == 6 for o in outs)
    assert e.kv.free_pages == 20  # everything freed


def test_prefix_reuse_matches_fresh(tiny):
    """A multi-turn conversation with KV prefix reuse: turn 1 (no cache)
    must equal a fresh run exactly; later turns are deterministic and
    reuse the cache.  Exact cross-path token equality for cached turns is
    NOT a bf16 invariant — the cached prefix KV was computed in a
    different prefill batch shape than a fresh full prefill, and rocBLAS
    rounding may legally flip a greedy argmax — so the cached turns
    assert determinism + reuse accounting instead."""
    from quickstart_streaming_agents_amd.models.serve import Engine, EngineLLM
    turn1 = "system prompt here\nuser question about prices"
    turn2 = turn1 + "\n[observation from http_get] competitor page says $209"
    turn3 = turn2 + "\n[observation from send_email] email sent ok"

    e_fresh = Engine(tiny, max_batch=4, max_seq_len=512)
    llm_fresh = EngineLLM(e_fresh)
    fresh = [llm_fresh([t], [8])[0] for t in (turn1, turn2, turn3)]

    convs = []
    for _ in range(2):
        e_conv = Engine(tiny, max_batch=4, max_seq_len=512)
        llm_conv = EngineLLM(e_conv)
        conv = [llm_conv([t], [8], ["c0"])[0] for t in (turn1, turn2, turn3)]
        llm_conv.release("c0")
        convs.append(conv)
    assert convs[0] == convs[1]          # cached decode is deterministic
    assert fresh[0] == convs[0][0]       # turn 1: no cache, exact match
    assert e_conv.stats.cached_prefix_tokens > 0  # reuse actually happened
    assert e_conv.stats.prefill_tokens < e_fresh.stats.prefill_tokens
    assert e_conv.kv.free_pages == e_conv.kv.n_pages


def test_batched_prefill_matches_single(tiny):
    """forward_prefill_batch over several sequences == per-sequence calls."""
    import torch as T
    prompts = [[1, 5, 9, 200, 17, 88], [1, 77, 31, 4], [1, 2, 3]]
    kv_a = tiny.new_kv_cache(16)
    items = []
    for sid, p in enumerate(prompts):
        kv_a.allocate(sid, len(p))
        items.append((T.tensor(p, dtype=T.int64, device="cuda:0"), sid, 0))
    batch_logits = tiny.forward_prefill_batch(items, kv_a)
    for sid, p in enumerate(prompts):
        kv_b = tiny.new_kv_cache(16)
        kv_b.allocate(0, len(p))
        solo = tiny.forward_prefill(
            T.tensor(p, dtype=T.int64, device="cuda:0"), kv_b, 0)
        T.testing.assert_close(batch_logits[sid], solo, atol=5e-2, rtol=5e-2)
        assert int(batch_logits[sid].argmax()) == int(solo.argmax())


def test_encoder_contract():
    from quickstart_streaming_agents_amd.models.encoder import EmbeddingEncoder
    enc = EmbeddingEncoder(device="cuda:0")
    texts = ["How do I create a Flink table?",
             "How do I create a Flink table now?",
             "boats dispatched to the French Quarter surge"]
    out = enc.embed_batch(texts)
    assert out.shape == (3, 1536)
    norms = np.linalg.norm(out, axis=1)
    assert np.allclose(norms, 1.0, atol=1e-3)
    # deterministic
    out2 = enc.embed_batch(texts)
    assert np.allclose(out, out2, atol=1e-5)
    # token overlap drives similarity
    sim01 = float(out[0] @ out[1])
    sim02 = float(out[0] @ out[2])
    assert sim01 > sim02


def test_gpu_vector_index_matches_cpu():
    """VectorIndex.search on GPU kernel == CPU numpy reference."""
    from quickstart_streaming_agents_amd.ops import ext
    from quickstart_streaming_agents_amd.vector.index import (HashingEmbedder,
                                                              VectorIndex)
    e = ext()
    emb = HashingEmbedder()
    idx = VectorIndex()
    rng = np.random.default_rng(0)
    for i in range(5000):
        v = rng.normal(size=1536).astype(np.float32)
        idx.add(f"D{i}", f"chunk {i}", v)
    q = rng.normal(size=(4, 1536)).astype(np.float32)
    qn = q / np.linalg.norm(q, axis=1, keepdims=True)
    docs_t = idx.to_torch("cuda:0")
    q_t = torch.from_numpy(qn).to("cuda:0")
    s, ids = e.topk_cosine(q_t, docs_t, 3)
    for row in range(4):
        hits = idx.search(qn[row], 3)
        assert [h.document_id for h in hits] == \
               [idx.ids[int(i)] for i in ids[row].tolist()]
        assert np.allclose(s[row].cpu().numpy(),
                           [h.score for h in hits], atol=1e-4)


def test_mixtral_gpu_engine():
    """tiny-moe Mixtral decodes on the HIP path (paged attention + routed
    experts) deterministically; CPU dispatch reference produces the same
    routing decisions for the first forward."""
    from quickstart_streaming_agents_amd.models.mixtral import (MixtralConfig,
                                                                MixtralModel)
    from quickstart_streaming_agents_amd.models.serve import Engine
    model = MixtralModel(MixtralConfig.preset("tiny-moe"), device="cuda:0",
                         seed=5)
    eng = Engine(model, max_batch=4, max_seq_len=256)
    outs = eng.generate_batch([[1, 5, 9, 13], [2, 4, 6]], [6, 6])
    assert all(len(o) == 6 for o in outs)
    eng2 = Engine(model, max_batch=4, max_seq_len=256)
    assert eng2.generate_batch([[1, 5, 9, 13], [2, 4, 6]], [6, 6]) == outs


def test_vector_index_gpu_search_matches_cpu():
    import numpy as np
    from quickstart_streaming_agents_amd.vector.index import (HashingEmbedder,
                                                              VectorIndex)
    emb = HashingEmbedder()
    idx = VectorIndex()
    rng = np.random.default_rng(11)
    for i in range(300):
        words = " ".join(rng.choice(
            ["window", "join", "agent", "kafka", "state"], size=5).tolist())
        idx.add(f"d{i}", words, emb.embed(words))
    queries = np.stack([emb.embed("agent state window"),
                        emb.embed("kafka join")])
    cpu = idx.search_batch(queries, 3)
    gpu = idx.search_batch_gpu(queries, 3, device="cuda:0")
    for c_hits, g_hits in zip(cpu, gpu):
        # duplicate chunks tie on score; compare the score vectors and
        # require every returned doc to actually carry its claimed score
        for c, g in zip(c_hits, g_hits):
            assert abs(c.score - g.score) < 1e-4
        assert {h.document_id for h in g_hits} <= set(idx.ids)


@pytest.mark.parametrize("rows,queries,k", [
    (40_000, 17, 3), (40_000, 37, 16), (40_000, 38, 16), (500, 16, 17),
    (500, 200, 5)])
def test_vector_index_batches(rows, queries, k):
    """The kernel and the matmul on either side of the rule between them; 40
    numbers a row, so a score's error stays under 40 roundings of f32."""
    import numpy as np
    from quickstart_streaming_agents_amd.vector.index import VectorIndex
    rng = np.random.default_rng(rows + queries)
    m = rng.standard_normal((rows, 40)).astype(np.float32)
    m /= np.linalg.norm(m, axis=1, keepdims=True)
    idx = VectorIndex(dim=40)
    idx._vecs, idx.metadata = list(m), [{}] * rows
    idx.ids = [str(i) for i in range(rows)]
    idx.chunks = idx.ids
    q = rng.standard_normal((queries, 40)).astype(np.float32)
    q[3] = m[rows - 1]
    want = q.astype(np.float64)
    want /= np.linalg.norm(want, axis=1, keepdims=True)
    want = want @ m.astype(np.float64).T
    tol = 40 * 2.0 ** -24
    for i, hits in enumerate(idx.search_batch_gpu(q, k, device="cuda:0")):
        top = np.sort(want[i])[::-1][:k]
        assert len(hits) == k and len({h.document_id for h in hits}) == k
        for h, best in zip(hits, top):
            assert abs(h.score - best) < tol
            assert abs(h.score - want[i, int(h.document_id)]) < tol
    q[5] = np.nan                      # a query without an answer
    hits = idx.search_batch_gpu(q, k, device="cuda:0")
    assert all(np.isnan(h.score) for h in hits[5]) and \
        hits[3][0].document_id == str(rows - 1)


@pytest.mark.parametrize("queries", [1, 15, 16])
def test_vector_index_beyond_the_kernel(queries):
    """More hits than the kernel keeps, a query that is not a number and
    documents without a score, for every number of queries."""
    import numpy as np
    from quickstart_streaming_agents_amd.vector.index import VectorIndex
    rng = np.random.default_rng(queries)
    m = rng.standard_normal((50, 8)).astype(np.float32)
    m /= np.linalg.norm(m, axis=1, keepdims=True)
    idx = VectorIndex(dim=8)
    idx._vecs, idx.metadata = list(m), [{}] * 50
    idx.ids = [str(i) for i in range(50)]
    idx.chunks = idx.ids
    q = m[:queries].copy()
    want = q.astype(np.float64) @ m.astype(np.float64).T
    for i, hits in enumerate(idx.search_batch_gpu(q, 17, device="cuda:0")):
        assert [h.document_id for h in hits] == \
            [str(j) for j in np.argsort(-want[i])[:17]]
    q[0] = np.nan
    assert all(np.isnan(h.score) for h in
               idx.search_batch_gpu(q, 3, device="cuda:0")[0])
    short = VectorIndex(dim=8)
    short._vecs = [m[0], np.full(8, np.nan, np.float32), m[1]]
    short.ids = short.chunks = ["a", "b", "c"]
    short.metadata = [{}] * 3
    for hits in short.search_batch_gpu(m[:queries], 3, device="cuda:0"):
        assert sorted(h.document_id for h in hits) == ["a", "c"]


def test_lab3_lab4_gpu_anomaly_matches_cpu_and_invariants():
    """The batched GPU anomaly path must reproduce the sequential CPU
    reference on the real lab datagen — and hence the determinism
    contracts (French Quarter only / Naples only)."""
    from quickstart_streaming_agents_amd.labs import datagen, pipelines
    from quickstart_streaming_agents_amd.wire import Broker

    b1 = Broker()
    datagen.publish_lab3(b1, seed=42)
    rows = pipelines.lab3_anomalies(b1)      # GPU path (cuda available)
    assert 1 <= len(rows) <= 2
    assert all(r["pickup_zone"] == "French Quarter" for r in rows)

    b2 = Broker()
    datagen.publish_lab4(b2, seed=42)
    rows4 = pipelines.lab4_anomalies(b2)
    assert [r["city"] for r in rows4] == ["Naples"]


def test_sql_driven_lab1_on_gpu_engine():
    """Catalog-driven lab1 runs end-to-end with the real decode engine on
    the GPU (tiny preset): content invariants hold with actual LLM decode
    in the loop."""
    from quickstart_streaming_agents_amd.agents.mcp import StubMcpServer
    from quickstart_streaming_agents_amd.labs.deploy import Deployment
    dep = Deployment(labs=(1,), device="cuda:0", model="tiny")
    dep.datagen(1)
    srv = StubMcpServer().start()
    try:
        rows = dep.run(1, mcp_server=srv)
    finally:
        srv.stop()
    assert len(rows) == 10
    assert all(r["agent_status"] == "SUCCESS" for r in rows)
    assert any(r["decision"] == "PRICE_MATCH" for r in rows)


def test_sql_driven_lab3_on_gpu_stack():
    """Lab3 end-to-end on the GPU stack: batched HIP anomaly scoring, the
    on-GPU embedding encoder, the HBM-resident index (GPU top-k), and the
    tiny decode engine — French Quarter contract preserved."""
    import json

    from quickstart_streaming_agents_amd.agents.mcp import StubMcpServer
    from quickstart_streaming_agents_amd.labs.deploy import Deployment
    dep = Deployment(labs=(3,), device="cuda:0", model="tiny")
    dep.datagen(3)
    srv = StubMcpServer().start()
    try:
        rows = dep.run(3, mcp_server=srv)
    finally:
        srv.stop()
    assert 1 <= len(rows) <= 2
    assert all(r["pickup_zone"] == "French Quarter" for r in rows)
    boats = json.loads(rows[0]["dispatch_json"])["boats"]
    assert 0 < len(boats) <= 8


def test_gpu_window_rows_match_cpu_assigner():
    """Columnar decode + HIP window_agg produces exactly the CPU
    TumblingWindows rows on the lab3 stream."""
    from quickstart_streaming_agents_amd.labs import datagen, schemas
    from quickstart_streaming_agents_amd.labs.pipelines import (
        MIN5_MS, _window_rows_gpu)
    from quickstart_streaming_agents_amd.runtime.windows import (
        TumblingWindows, aggregate)
    from quickstart_streaming_agents_amd.wire import AvroConsumer, Broker
    b = Broker()
    datagen.publish_lab3(b, seed=42)
    gpu_rows = _window_rows_gpu(b, "ride_requests", schemas.RIDE_REQUESTS,
                                "request_ts", "pickup_zone", MIN5_MS)
    rides = [r for _, r in AvroConsumer(b, "ride_requests",
                                        schemas.RIDE_REQUESTS).poll()]
    tw = TumblingWindows(MIN5_MS, lambda r: r["pickup_zone"],
                         lambda r: r["request_ts"], watermark_delay_ms=5000)
    cpu_rows = aggregate(tw.feed(rides) + tw.flush(),
                         {"request_count": len})
    cpu_rows.sort(key=lambda r: (r["window_start"], r["key"]))
    assert [(r["key"], r["window_start"], r["request_count"])
            for r in gpu_rows] == \
        [(r["key"], r["window_start"], r["request_count"])
         for r in cpu_rows]


def test_generic_sql_executor_on_gpu_engine():
    """The generic CTAS executor (sql/exec.py) drives the REAL GPU stack:
    EngineLLM decode, on-GPU embedding encoder, HBM-resident index —
    lab3's French Quarter contract holds end-to-end through generic SQL
    execution (CPU equivalence is tests/test_sql_exec.py)."""
    from quickstart_streaming_agents_amd.agents.mcp import StubMcpServer
    from quickstart_streaming_agents_amd.labs.deploy import Deployment
    dep = Deployment(labs=(3,), device="cuda:0", model="tiny")
    dep.datagen(3)
    srv = StubMcpServer().start()
    try:
        rows = dep.run_sql(3, mcp_server=srv)
    finally:
        srv.stop()
    assert 1 <= len(rows) <= 2
    assert all(r["pickup_zone"] == "French Quarter" for r in rows)
    assert all(r["api_response"] for r in rows)


def test_serve_api_on_gpu_engine():
    """The HTTP serving surface (serve_api.py) wired to the REAL GPU
    stack: EngineLLM completions, GPU embedder + HBM index search, and
    an agent episode — all through the FastAPI app."""
    import pytest as _pytest
    _pytest.importorskip("fastapi")
    from fastapi.testclient import TestClient

    from quickstart_streaming_agents_amd.serve_api import build_lab_app
    app = build_lab_app(device="cuda:0", model="tiny", labs=(1, 2))
    try:
        with TestClient(app) as c:
            out = c.post("/v1/completions",
                         json={"prompt": "hello", "max_tokens": 8}).json()
            assert out["choices"][0]["text"]
            emb = c.post("/v1/embeddings", json={"input": "x"}).json()
            assert emb["dims"] == 1536
            hits = c.post("/v1/search",
                          json={"query": "How do I create a Flink table?",
                                "k": 2}).json()["hits"]
            assert len(hits) == 2 and hits[0]["score"] >= hits[1]["score"]
            ag = c.post("/v1/agents/price_match_agent",
                        json={"prompt": "check AirPods"}).json()
            assert ag["status"] in ("SUCCESS", "FAILED")
            assert "qsa_requests_total" in c.get("/metrics").text
    finally:
        app.state.mcp_server.stop()


def test_qwen_bias_engine_on_gpu():
    """Qwen2-family decode (qkv biases) through the full GPU engine:
    hipGraph capture with the bias add in the captured region, greedy
    decode deterministic across two engines."""
    from quickstart_streaming_agents_amd.models.llama import (LlamaConfig,
                                                              LlamaModel)
    from quickstart_streaming_agents_amd.models.serve import Engine
    cfg = LlamaConfig.preset("tiny-qwen")
    outs = []
    for _ in range(2):
        eng = Engine(LlamaModel(cfg, device="cuda:0", seed=13),
                     max_batch=4, max_seq_len=256)
        outs.append(eng.generate_batch([[3, 7, 11], [2, 9, 4, 6]], [6, 6]))
    assert outs[0] == outs[1]
    assert all(len(o) == 6 for o in outs[0])


def test_rccl_all_reduce_inside_hipgraph():
    """RCCL-in-graph validation: a TP-sharded decode
    step whose per-layer all-reduce is RECORDED into the hipGraph must
    replay identically to the eager path.  World=1 nccl(=RCCL) group on
    the lease box: the collective still goes through the RCCL enqueue
    path that capture must record."""
    import os
    import torch.distributed as dist
    from quickstart_streaming_agents_amd.models.llama import (LlamaConfig,
                                                              LlamaModel)
    from quickstart_streaming_agents_amd.models.serve import Engine
    created = False
    if not dist.is_initialized():
        os.environ.setdefault("MASTER_ADDR", "127.0.0.1")
        os.environ.setdefault("MASTER_PORT", "29511")
        dist.init_process_group("nccl", rank=0, world_size=1)
        created = True
    try:
        cfg = LlamaConfig.preset("tiny")
        # tp_size=2/rank 0 shards the weights; the TP group holds only
        # this rank, so the all-reduce is a world-1 RCCL collective.
        model = LlamaModel(cfg, device="cuda:0", seed=5, tp_rank=0,
                           tp_size=2, tp_group=dist.group.WORLD)
        prompts = [[3, 7, 11, 19], [2, 9, 4, 6, 8]]

        # max_batch == n prompts: the graph decodes exactly the same
        # GEMM shapes as eager (padding rows change bf16 numerics)
        eng_g = Engine(model, max_batch=2, max_seq_len=256)
        assert eng_g.use_graph
        out_g = eng_g.generate_batch([list(p) for p in prompts], [8, 8])
        assert eng_g._graph is not None, \
            "graph capture must succeed with RCCL in the captured region"

        eng_e = Engine(model, max_batch=2, max_seq_len=256)
        eng_e.use_graph = False
        out_e = eng_e.generate_batch([list(p) for p in prompts], [8, 8])
        assert out_g == out_e
    finally:
        if created:
            dist.destroy_process_group()


def test_rccl_collectives_on_hardware():
    """Exercise every collective the TP/EP paths use through RCCL on the
    device (world=1): all_reduce, all_to_all_single, all_gather,
    broadcast — shapes/dtypes as the model paths issue them."""
    import os
    import torch.distributed as dist
    created = False
    if not dist.is_initialized():
        os.environ.setdefault("MASTER_ADDR", "127.0.0.1")
        os.environ.setdefault("MASTER_PORT", "29512")
        dist.init_process_group("nccl", rank=0, world_size=1)
        created = True
    try:
        dev = "cuda:0"
        x = torch.randn(24, 256, device=dev, dtype=torch.bfloat16)
        y = x.clone()
        dist.all_reduce(y)
        assert torch.equal(x, y)
        # EP token shuffle (parallel/ep.py all_to_all_single with splits)
        t = torch.randn(17, 64, device=dev, dtype=torch.bfloat16)
        out = torch.empty_like(t)
        dist.all_to_all_single(out, t, [17], [17])
        assert torch.equal(out, t)
        gathered = [torch.empty_like(x)]
        dist.all_gather(gathered, x)
        assert torch.equal(gathered[0], x)
        dist.broadcast(x, src=0)
        torch.cuda.synchronize()
    finally:
        if created:
            dist.destroy_process_group()


def test_encoder_mfma_attention_matches_bmm_reference():
    """K1 encoder bidirectional varlen MFMA attention (CAUSAL=false
    paged_attn_prefill) vs the padded-bmm reference ON THE SAME DEVICE
    AND DTYPE — only the attention implementation differs (an f32-CPU
    end-to-end comparison through 12 random layers diverges chaotically
    from bf16 rounding alone and tests nothing).  VERDICT r1 item 7."""
    from quickstart_streaming_agents_amd.models.encoder import (
        EmbeddingEncoder, EncoderConfig)
    cfg = EncoderConfig(n_layers=4)
    enc = EmbeddingEncoder(cfg, device="cuda:0", seed=2)
    texts = ["How do I create a Flink table?",
             "a much longer document about insurance claims in Naples "
             "Florida with anomalous totals across a six hour window " * 4,
             "x",
             "boats dispatched to the French Quarter surge zone"]
    out_hip = enc.embed_batch(texts)
    enc._use_hip = False
    out_bmm = enc.embed_batch(texts)
    assert out_hip.shape == out_bmm.shape == (4, 1536)
    assert np.isfinite(out_hip).all(), \
        f"hip path non-finite rows: {(~np.isfinite(out_hip).all(1)).nonzero()}"
    assert np.isfinite(out_bmm).all(), \
        f"bmm path non-finite rows: {(~np.isfinite(out_bmm).all(1)).nonzero()}"
    for i in range(4):
        cos = float(out_hip[i] @ out_bmm[i])
        assert cos > 0.98, f"text {i}: cosine {cos}"


def test_encoder_varlen_batch_invariance():
    """Embedding of a text must not depend on what else is in the batch
    (varlen kernel correctness under ragged batching)."""
    from quickstart_streaming_agents_amd.models.encoder import (
        EmbeddingEncoder, EncoderConfig)
    enc = EmbeddingEncoder(EncoderConfig(n_layers=4), device="cuda:0",
                           seed=4)
    t = "the quick brown fox jumps over the lazy dog"
    alone = enc.embed_batch([t])[0]
    mixed = enc.embed_batch(
        ["padding " * 60, t, "short"])[1]
    cos = float(alone @ mixed)
    assert cos > 0.999, cos


def test_full_size_llama3_8b_engine():
    """Engine-level GPU test at the FLAGSHIP size (llama3-8b, 32 layers,
    128256 vocab): graph decode == eager decode at matched batch shapes,
    real decode-shape kernels (fp8 skinny / paged attention) on the hot
    path.  (engine-level GPU tests exercised a 256-hidden
    toy; this closes that gap.)"""
    from quickstart_streaming_agents_amd.models import build_model
    from quickstart_streaming_agents_amd.models.serve import Engine
    model = build_model("llama3-8b", device="cuda:0")
    assert model.use_fp8 and "wgu_f8" in model.layers[0]
    prompts = [[1] + list(range(100, 160)), [1] + list(range(300, 340))]
    eng_g = Engine(model, max_batch=2, max_seq_len=512)
    out_g = eng_g.generate_batch([list(p) for p in prompts], [12, 12])
    assert eng_g._graph is not None
    eng_e = Engine(model, max_batch=2, max_seq_len=512)
    eng_e.use_graph = False
    out_e = eng_e.generate_batch([list(p) for p in prompts], [12, 12])
    assert out_g == out_e
    assert all(len(o) == 12 for o in out_g)
    # all tokens inside the vocab
    assert all(0 <= t < 128256 for o in out_g for t in o)


def test_stream_pipeline_gpu_matches_sequential():
    """StreamPipeline on real HIP streams (one per stage, event-chained)
    == sequential execution; lab2 index build through the pipelined path
    == sequential add_documents."""
    from quickstart_streaming_agents_amd.runtime.streams import (
        StreamPipeline, pipelined_embed_index)
    torch.manual_seed(0)
    w1 = torch.randn(256, 256, device="cuda:0")
    w2 = torch.randn(256, 256, device="cuda:0")
    batches = [torch.randn(64, 256, device="cuda:0") for _ in range(12)]
    pipe = StreamPipeline([lambda x: x @ w1,
                           lambda x: torch.relu(x),
                           lambda x: x @ w2])
    assert pipe.use_streams
    got = pipe.run(batches)
    for b, g in zip(batches, got):
        ref = torch.relu(b @ w1) @ w2
        torch.testing.assert_close(g, ref)

    from quickstart_streaming_agents_amd.labs import datagen
    from quickstart_streaming_agents_amd.models.encoder import (
        EmbeddingEncoder, EncoderConfig)
    from quickstart_streaming_agents_amd.vector.index import VectorIndex
    enc = EmbeddingEncoder(EncoderConfig(n_layers=2), device="cuda:0",
                           seed=3)
    docs = [{"document_id": f"d{i}", "chunk": c["chunk"]}
            for i, c in enumerate(datagen.lab2_documents(n_chunks=24))]
    seq = VectorIndex()
    seq.add_documents([dict(d) for d in docs], enc)
    pip = VectorIndex()
    pipelined_embed_index(enc, pip, [dict(d) for d in docs], batch_size=5)
    q = enc.embed_batch(["anomaly windows in flink"])[0]
    assert [h.document_id for h in seq.search(q, 3)] == \
        [h.document_id for h in pip.search(q, 3)]


def test_generic_sql_lab1_model_driven_on_engine():
    """The GENERIC SQL executor runs lab1 end-to-end on the GPU engine
    with MODEL-DRIVEN agents (no scripted policies): grammar-constrained
    decisions through the real decode path, one result row per enriched
    order, status from the episode machine."""
    import torch as T
    T.manual_seed(99)
    from quickstart_streaming_agents_amd.agents.mcp import StubMcpServer
    from quickstart_streaming_agents_amd.labs.deploy import Deployment
    dep = Deployment(labs=(1,), device="cuda:0", model="tiny")
    dep.datagen(1)
    with StubMcpServer() as srv:
        ex = dep.sql_executor(1, mcp_server=srv, scripted_policies=False)
        rows = ex.run_table("price_match_results")
    assert len(rows) >= 1
    assert all(r["agent_status"] in ("SUCCESS", "FAILED") for r in rows)
    ids = [r["order_id"] for r in rows]
    assert len(ids) == len(set(ids))


def test_encoder_needs_one_module(monkeypatch):
    """qsa_hip alone serves the encoder; products in other tiles differ in the
    order of their f32 sums and in whether the gate is rounded before it acts."""
    from quickstart_streaming_agents_amd import ops
    from quickstart_streaming_agents_amd.models.encoder import EmbeddingEncoder
    enc = EmbeddingEncoder(device="cuda:0")
    for n in (1, 40):                    # a few rows, and beyond 2048
        texts = [f"ticket {i} about the harbor route " * 20 for i in range(n)]
        want = enc.embed_batch(texts)
        with monkeypatch.context() as m:
            m.setattr(ops, "_lm_ext", None)
            got = enc.embed_batch(texts)
        assert np.abs(got - want).max() <= 0.02 * np.abs(want).max()


def test_encoder_layers_at_once():
    """All layers in one call against the calls one by one: the same kernels, so the
    same numbers; weights that the one call does not take are left to the others."""
    from quickstart_streaming_agents_amd.models.encoder import (
        EmbeddingEncoder, EncoderConfig)
    enc = EmbeddingEncoder(EncoderConfig(n_layers=3), device="cuda:0", seed=4)
    for lens in ([1], [15], [33], [64, 65, 1], [130] * 9, [200] * 48):
        n = len(lens)
        g = torch.Generator().manual_seed(sum(lens))
        res = torch.randn(sum(lens), 384, generator=g).bfloat16().to("cuda:0")
        blocks = [(i, p) for i, m in enumerate(lens) for p in range(0, m, 64)]
        maps = [torch.tensor(x, dtype=torch.int32, device="cuda:0") for x in (
            [b[0] for b in blocks], [b[1] for b in blocks],
            [sum(lens[:i]) for i in range(n)], lens)]
        one, two = res.clone(), res.clone()
        got = enc._native_layers(one, *maps)
        want = enc._layers_by_call(two, *maps)
        assert got is not None and torch.equal(got, want)
        assert torch.equal(one, two)
    wqkv = enc.layers[1]["wqkv"]
    enc.layers[1]["wqkv"] = wqkv.t().contiguous().t()
    before = res.clone()
    assert enc._native_layers(res, *maps) is None
    assert torch.equal(res, before)


@pytest.mark.parametrize("rows", [32, 33, 130, 320])
def test_encoder_down_product(rows):
    """The feed-forward's second product and the norm that adds it: beyond 32
    rows in shares of K, which it adds sooner than a product is finished; either
    way rounded once, as it would be stored, before the residual is."""
    from quickstart_streaming_agents_amd.models.encoder import (
        EmbeddingEncoder, EncoderConfig)
    from quickstart_streaming_agents_amd.ops import dispatch as D
    enc = EmbeddingEncoder(EncoderConfig(n_layers=1), device="cuda:0", seed=4)
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, 1536, generator=g).bfloat16().to("cuda:0")
    w = enc.layers[0]["wdown"]
    y = enc._linear(x, w, parts=True)
    assert y.dim() == (2 if rows <= 32 else 3) and \
        y.dtype == (torch.bfloat16 if rows <= 32 else torch.float32)
    res = torch.randn(rows, 384, generator=g).bfloat16().to("cuda:0")
    old = res.double()
    D.rmsnorm_residual(y, res, enc.final_norm, 1e-5)
    want = x.double() @ w.double().T
    err = 1536 * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    # half an ulp of bf16 is up to 2^-8: of the product, and of the sum, which may
    # be larger by the product's
    assert ((res.double() - old - want).abs() <= 2.0 ** -8 * (
        1.01 * want.abs() + (old + want).abs()) + 1.01 * err).all()


def test_encoder_products_of_another(monkeypatch):
    """A product that is replaced, in a subclass or an object, is the one that
    runs, for every layer."""
    from quickstart_streaming_agents_amd.models.encoder import (
        EmbeddingEncoder, EncoderConfig)

    class Counted(EmbeddingEncoder):
        def _linear(self, x, w, glu=False, parts=False):
            calls.append(w.shape)
            return super()._linear(x, w, glu)

    calls, cfg, text = [], EncoderConfig(n_layers=2), ["water and light"]
    plain = EmbeddingEncoder(cfg, device="cuda:0", seed=4)
    want = plain.embed_batch(text)
    assert np.abs(Counted(cfg, device="cuda:0", seed=4).embed_batch(text) -
                  want).max() <= 0.02 * np.abs(want).max()
    assert len(calls) == 9                  # and the projection
    linear = plain._linear
    monkeypatch.setattr(plain, "_linear", lambda *a, **k: calls.append(0) or
                        linear(*a, **k))
    assert np.array_equal(plain.embed_batch(text), want)
    assert len(calls) == 18


@pytest.mark.parametrize("which", ["cos", "sin", 0, 1, 2, 3])
def test_encoder_layers_refuses_host_operands(which):
    """Tables and maps whose memory is the host's: an error before anything is
    launched."""
    from quickstart_streaming_agents_amd.models.encoder import (
        EmbeddingEncoder, EncoderConfig)
    enc = EmbeddingEncoder(EncoderConfig(n_layers=1), device="cuda:0", seed=4)
    maps = [torch.tensor(x, dtype=torch.int32, device="cuda:0")
            for x in ([0], [0], [0], [7])]
    if which in ("cos", "sin"):
        name = "rope_" + which
        setattr(enc, name, getattr(enc, name).cpu())
    else:
        maps[which] = maps[which].cpu()
    res = torch.randn(7, 384).bfloat16().to("cuda:0")
    before = res.clone()
    with pytest.raises(RuntimeError, match="operands must be on"):
        enc._native_layers(res, *maps)
    assert torch.equal(res, before)
