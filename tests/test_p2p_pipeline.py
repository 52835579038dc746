"""Decentralized pipeline over the loopback transport: 2/3-stage peer
executors produce the same greedy tokens as the single-process engine
(the reference's in-process pipeline emulation test strategy,
tests/test_executor.py analogue). Also: codec round-trip."""

import pytest
import torch

from parallax_amd.p2p import codec
from parallax_amd.p2p.peer_executor import PeerExecutor
from parallax_amd.p2p.transport import LoopbackTransport
from parallax_amd.server.request import IntermediateRequest
from parallax_amd.server.sampling_params import SamplingParams

from tests.test_pipeline_parallel import PROMPTS, full_state_dict, run_single_process, tiny_cfg


def test_codec_roundtrip():
    h = torch.randn(5, 64, dtype=torch.bfloat16)
    req = IntermediateRequest(
        rid="r1", routing_table=["a", "b"], current_position=7,
        num_new_tokens=5, is_prefill=True, hidden_states=h,
        sampling_params=SamplingParams(temperature=0.5, top_k=5),
        input_ids=[1, 2, 3, 4, 5],
    )
    msg = codec.decode(codec.encode_forward([req]))
    assert msg["kind"] == "forward"
    r = msg["reqs"][0]
    assert r.rid == "r1" and r.routing_table == ["a", "b"]
    assert r.current_position == 7 and r.is_prefill
    assert torch.equal(r.hidden_states, h)
    assert r.sampling_params.temperature == 0.5 and r.sampling_params.top_k == 5

    ctl = codec.decode(codec.encode_control("release", ["r1", "r2"]))
    assert ctl == {"kind": "release", "rids": ["r1", "r2"]}
    tok = codec.decode(codec.encode_tokens([("r1", 42)]))
    assert tok["kind"] == "token" and tok["tokens"][0] == ["r1", 42] or \
        tok["tokens"][0] == ("r1", 42)


@pytest.mark.parametrize("n_stages", [2, 3])
def test_loopback_pipeline_matches_single(n_stages):
    expected = run_single_process()
    cfg = tiny_cfg()
    registry = {}
    peer_ids = [f"peer{i}" for i in range(n_stages)]
    # contiguous layer split
    base, rem = divmod(cfg.num_layers, n_stages)
    spans, pos = [], 0
    for i in range(n_stages):
        n = base + (1 if i < rem else 0)
        spans.append((pos, pos + n))
        pos += n
    peers = []
    sd = full_state_dict(cfg)
    for pid, (s, e) in zip(peer_ids, spans):
        t = LoopbackTransport(pid, registry)
        px = PeerExecutor(cfg, s, e, pid, t, dtype=torch.float32,
                          num_kv_blocks=128, block_size=8)
        for name, w in sd.items():
            px.model.load_hf_weight(name, w)
        peers.append(px)

    head = peers[0]
    sp = SamplingParams(temperature=0.0, max_new_tokens=6, ignore_eos=True)
    rids = [head.submit(p, sp, peer_ids) for p in PROMPTS]
    outputs = {rid: [] for rid in rids}
    done = set()
    for _ in range(2000):
        for px in peers:
            px.step(recv_timeout=0.001)
        for out in head.drain_outputs():
            outputs[out.rid].append(out.token_id)
            if out.finished:
                done.add(out.rid)
        if len(done) == len(rids):
            break
    assert [outputs[r] for r in rids] == expected
    # release control packets freed downstream cache state
    for _ in range(20):
        for px in peers:
            px.step(recv_timeout=0.001)
    for px in peers[1:]:
        assert not px._peer_positions


def test_tcp_transport_roundtrip():
    from parallax_amd.p2p.transport import TcpTransport

    a = TcpTransport("a", "127.0.0.1", 0)
    b = TcpTransport("b", "127.0.0.1", 0)
    a.set_peer_addr("b", "127.0.0.1", b.port)
    b.set_peer_addr("a", "127.0.0.1", a.port)
    a.send("b", b"hello" * 1000)
    got = b.recv(timeout=5)
    assert got == b"hello" * 1000
    b.send("a", b"pong")
    assert a.recv(timeout=5) == b"pong"
    a.close()
    b.close()


def _run_p2p(cfg, sd, n_stages, prompts, n_new=5):
    registry = {}
    peer_ids = [f"peer{i}" for i in range(n_stages)]
    base, rem = divmod(cfg.num_layers, n_stages)
    spans, pos = [], 0
    for i in range(n_stages):
        n = base + (1 if i < rem else 0)
        spans.append((pos, pos + n))
        pos += n
    peers = []
    for pid, (s, e) in zip(peer_ids, spans):
        t = LoopbackTransport(pid, registry)
        px = PeerExecutor(cfg, s, e, pid, t, dtype=torch.float32,
                          num_kv_blocks=128, block_size=8)
        for name, w in sd.items():
            px.model.load_hf_weight(name, w)
        if hasattr(px.model, "finalize_weights"):
            px.model.finalize_weights()
        peers.append(px)
    head = peers[0]
    sp = SamplingParams(temperature=0.0, max_new_tokens=n_new, ignore_eos=True)
    rids = [head.submit(p, sp, peer_ids) for p in prompts]
    outputs = {rid: [] for rid in rids}
    done = set()
    for _ in range(3000):
        for px in peers:
            px.step(recv_timeout=0.001)
        for out in head.drain_outputs():
            outputs[out.rid].append(out.token_id)
            if out.finished:
                done.add(out.rid)
        if len(done) == len(rids):
            break
    return [outputs[r] for r in rids]


def test_p2p_hybrid_linear_stack():
    """Qwen3-Next-style hybrid (deltanet + attention) over 2 peers: linear
    state slots live per peer and must reproduce the single-engine output."""
    import transformers

    from parallax_amd.models import get_model_class
    from parallax_amd.models.config import ModelConfig
    from parallax_amd.server.engine import Engine, EngineArgs

    torch.manual_seed(41)
    hf_cfg = transformers.Qwen3NextConfig(
        vocab_size=128, hidden_size=64, intermediate_size=128,
        moe_intermediate_size=32, shared_expert_intermediate_size=32,
        num_hidden_layers=4, num_attention_heads=4, num_key_value_heads=2,
        head_dim=32, num_experts=4, num_experts_per_tok=2, norm_topk_prob=True,
        decoder_sparse_step=1, mlp_only_layers=[],
        linear_num_key_heads=2, linear_num_value_heads=4,
        linear_key_head_dim=16, linear_value_head_dim=16,
        linear_conv_kernel_dim=4,
        layer_types=["linear_attention", "full_attention"] * 2,
        max_position_embeddings=512, tie_word_embeddings=False,
        rope_parameters={"rope_type": "default", "rope_theta": 10000.0,
                         "partial_rotary_factor": 0.25},
    )
    hf = transformers.Qwen3NextForCausalLM(hf_cfg).eval()
    cfg = ModelConfig.from_hf_config(
        hf_cfg.to_dict() | {"architectures": ["Qwen3NextForCausalLM"]}
    )
    prompts = [[7, 42, 99, 5, 81, 23], [3, 9, 27]]
    sd = dict(hf.state_dict())
    # single-engine baseline
    eng = Engine(cfg, EngineArgs(block_size=8, num_kv_blocks=128,
                                 dtype=torch.float32, max_batch_size=8))
    m = get_model_class(cfg.architecture)(cfg).eval()
    for name, w in sd.items():
        m.load_hf_weight(name, w)
    eng.model = m.float()
    sp = SamplingParams(temperature=0.0, max_new_tokens=5, ignore_eos=True)
    expect = list(eng.generate(prompts, [sp] * 2).values())
    got = _run_p2p(cfg, sd, 2, prompts)
    assert got == expect


def test_p2p_abort_releases_downstream():
    """Head-side abort mid-generation: the client stream gets a terminator
    PeerOutput (token_id -1) and the downstream peer's cache state is
    released via the broadcast."""
    cfg = tiny_cfg()
    registry = {}
    sd = full_state_dict(cfg)
    peers = []
    for pid, (s, e) in zip(["h", "t"], [(0, 2), (2, 4)]):
        t = LoopbackTransport(pid, registry)
        px = PeerExecutor(cfg, s, e, pid, t, dtype=torch.float32,
                          num_kv_blocks=128, block_size=8)
        for name, w in sd.items():
            px.model.load_hf_weight(name, w)
        peers.append(px)
    head, tail = peers
    sp = SamplingParams(temperature=0.0, max_new_tokens=64, ignore_eos=True)
    rid = head.submit([1, 2, 3, 4], sp, ["h", "t"])
    toks = []
    finished = None
    for i in range(400):
        for px in peers:
            px.step(recv_timeout=0.001)
        for out in head.drain_outputs():
            if out.token_id >= 0:
                toks.append(out.token_id)
            if out.finished:
                finished = out
        if len(toks) >= 5 and finished is None:
            head.abort(rid)
        if finished is not None:
            # let release broadcasts drain
            for _ in range(20):
                for px in peers:
                    px.step(recv_timeout=0.001)
            break
    assert finished is not None and finished.finish_reason == "abort"
    assert 5 <= len(toks) < 64
    assert rid not in tail._peer_positions  # downstream state released


def test_codec_large_tensor_and_empty_batch():
    """Wire codec edge cases: multi-MB bf16 hidden states round-trip intact;
    empty forward batches survive."""
    h = torch.randn(2048, 1024, dtype=torch.bfloat16)
    req = IntermediateRequest(
        rid="big", routing_table=["a"], current_position=0,
        num_new_tokens=2048, is_prefill=True, hidden_states=h,
    )
    msg = codec.decode(codec.encode_forward([req]))
    assert torch.equal(msg["reqs"][0].hidden_states, h)
    empty = codec.decode(codec.encode_forward([]))
    assert empty["kind"] == "forward" and empty["reqs"] == []


def test_tcp_transport_many_frames_in_order():
    from parallax_amd.p2p.transport import TcpTransport

    a = TcpTransport("a", "127.0.0.1", 0)
    b = TcpTransport("b", "127.0.0.1", 0)
    a.set_peer_addr("b", "127.0.0.1", b.port)
    payloads = [bytes([i]) * (1000 * (i + 1)) for i in range(20)]
    for p in payloads:
        a.send("b", p)
    got = []
    for _ in range(20):
        got.append(b.recv(timeout=5))
    assert got == payloads
    a.close()
    b.close()


def test_tcp_auth_handshake():
    """Auth-token transports accept matching peers and drop mismatched or
    unauthenticated connections."""
    import time as _time

    from parallax_amd.p2p.transport import TcpTransport

    a = TcpTransport("a", host="127.0.0.1", auth_token="s3cret")
    b = TcpTransport("b", host="127.0.0.1", auth_token="s3cret")
    bad = TcpTransport("x", host="127.0.0.1", auth_token="wrong")
    naked = TcpTransport("n", host="127.0.0.1")  # no token at all
    try:
        a.set_peer_addr("b", "127.0.0.1", b.port)
        bad.set_peer_addr("b", "127.0.0.1", b.port)
        naked.set_peer_addr("b", "127.0.0.1", b.port)
        a.send("b", b"hello")
        assert b.recv(timeout=5.0) == b"hello"
        bad.send("b", b"evil")
        naked.send("b", b"sneaky")
        assert b.recv(timeout=0.8) is None  # both rejected at handshake
    finally:
        for t in (a, b, bad, naked):
            t.close()


def test_dead_peer_aborts_requests_not_node():
    """A routing table naming a nonexistent peer must terminate the affected
    streams (abort) instead of crashing the head or hanging the client."""
    cfg = tiny_cfg()
    registry = {}
    t = LoopbackTransport("head", registry)
    head = PeerExecutor(cfg, 0, cfg.num_layers // 2, "head", t,
                        dtype=torch.float32, num_kv_blocks=128, block_size=8)
    for name, w in full_state_dict(cfg).items():
        head.model.load_hf_weight(name, w)
    sp = SamplingParams(temperature=0.0, max_new_tokens=4, ignore_eos=True)
    rid = head.submit([5, 9, 13], sp, ["head", "ghost-peer"])
    finished = []
    for _ in range(200):
        head.step(recv_timeout=0.001)  # must not raise
        finished += [o for o in head.drain_outputs() if o.finished]
        if finished:
            break
    assert finished and finished[0].rid == rid
    assert finished[0].finish_reason == "abort"
    # head keeps serving: nothing left running
    assert not head.scheduler.running


def test_head_frontend_stream_stop_string():
    """The WAN head's SSE path truncates at a stop string and aborts the
    executor request (fake agent, no network)."""
    import asyncio

    fastapi = pytest.importorskip("fastapi")
    from fastapi.testclient import TestClient

    from parallax_amd.p2p.head_frontend import create_head_app
    from parallax_amd.p2p.peer_executor import PeerOutput
    from parallax_amd.server.tokenizer_util import TokenizerWrapper

    aborted = []

    class FakeExec:
        def abort(self, rid):
            aborted.append(rid)

    class FakeAgent:
        node_id = "head"
        executor = FakeExec()

        def submit(self, prompt_ids, sp, routing, aio_loop=None,
                   aio_queue=None):
            # feed 5 tokens then a terminator into the asyncio queue
            for i, t in enumerate([10, 11, 12, 13, 14]):
                aio_loop.call_soon_threadsafe(
                    aio_queue.put_nowait,
                    PeerOutput("r1", t, i == 4,
                               "length" if i == 4 else None))
            aio_loop.call_soon_threadsafe(aio_queue.put_nowait, None)
            return "r1", aio_queue

    tok = TokenizerWrapper(vocab_size=64)
    app = create_head_app(FakeAgent(), tok, "fake")
    with TestClient(app) as c:
        stop = tok.decode([12])  # third token's text
        text, finish = "", None
        with c.stream("POST", "/v1/chat/completions", json={
            "messages": [{"role": "user", "content": "x"}],
            "max_tokens": 5, "stream": True, "stop": [stop],
        }) as r:
            import json as _json

            for line in r.iter_lines():
                if not line.startswith("data: ") or line == "data: [DONE]":
                    continue
                msg = _json.loads(line[6:])
                for ch in msg.get("choices", []):
                    text += (ch.get("delta") or {}).get("content") or ""
                    if ch.get("finish_reason"):
                        finish = ch["finish_reason"]
    assert finish == "stop"
    assert stop not in text
    assert aborted == ["r1"]


try:
    from hypothesis import HealthCheck, given, settings
    from hypothesis import strategies as st
    _HYP = True
except ImportError:  # pragma: no cover
    _HYP = False


@pytest.mark.skipif(not _HYP, reason="hypothesis not installed")
@settings(max_examples=40, deadline=None,
          suppress_health_check=[HealthCheck.too_slow])
@given(rows=st.integers(min_value=0, max_value=9),
       cols=st.integers(min_value=1, max_value=33),
       pos=st.integers(min_value=0, max_value=100000),
       tok=st.integers(min_value=-1, max_value=200000),
       temp=st.sampled_from([0.0, 0.7, 1.0]),
       prefill=st.booleans())
def test_codec_roundtrip_property(rows, cols, pos, tok, temp, prefill):
    """Wire codec: arbitrary packet shapes survive encode/decode exactly
    (hidden-state bytes, positions, token ids, sampling params)."""
    from parallax_amd.p2p import codec
    from parallax_amd.server.request import IntermediateRequest
    from parallax_amd.server.sampling_params import SamplingParams

    h = torch.randn(rows, cols) if rows else None
    pkt = IntermediateRequest(
        rid="x" * 8, current_position=pos, hidden_states=h,
        next_token_id=tok if tok >= 0 else None,
        routing_table=["a", "b"], is_prefill=prefill,
        num_new_tokens=max(1, rows),
        sampling_params=SamplingParams(temperature=temp, max_new_tokens=5),
    )
    out = codec.decode(codec.encode_forward([pkt]))
    assert out["kind"] == "forward"
    got = out["reqs"][0]
    assert got.rid == pkt.rid and got.current_position == pos
    assert got.next_token_id == pkt.next_token_id
    assert got.is_prefill == prefill
    assert got.sampling_params.temperature == temp
    if h is None:
        assert got.hidden_states is None or got.hidden_states.numel() == 0
    else:
        assert torch.equal(got.hidden_states, h)


def test_tcp_transport_survives_garbage():
    """Random bytes, oversized frame claims and wrong auth must not kill the
    accept loop or leak into the inbox."""
    import socket as sk
    import time as _time

    from parallax_amd.p2p.transport import TcpTransport

    t = TcpTransport("victim", host="127.0.0.1", port=0,
                     max_frame_bytes=1 << 20, auth_token="sekret")
    try:
        for payload in (b"\x00" * 3,                      # truncated header
                        b"\xff" * 12,                     # absurd frame length
                        b"AUTH" + (99999).to_bytes(4, "little") + b"x",
                        b"GARBAGEGARBAGE"):
            with sk.create_connection(("127.0.0.1", t.port), timeout=5) as c:
                c.sendall(payload)
                _time.sleep(0.05)
        # a well-formed authed frame still arrives after all that
        import struct

        with sk.create_connection(("127.0.0.1", t.port), timeout=5) as c:
            tok = b"sekret"
            c.sendall(b"AUTH" + struct.pack("<I", len(tok)) + tok)
            msg = b"hello"
            c.sendall(struct.pack("<Q", len(msg)) + msg)
            _time.sleep(0.2)
        got = t.recv(timeout=5)
        assert got == b"hello"
        assert t.recv(timeout=0.1) is None  # nothing from the garbage
    finally:
        t.close() if hasattr(t, "close") else None
