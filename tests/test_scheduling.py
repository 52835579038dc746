"""Cluster-scheduling tests with fabricated nodes (mirrors the reference's
tests/scheduler_tests strategy: the brain is pure logic, drive it with fake
hardware profiles and assert allocation/routing invariants)."""

import pytest

from parallax_amd.models.config import ModelConfig
from parallax_amd.scheduling.layer_allocation import (
    GreedyLayerAllocator,
    DynamicProgrammingLayerAllocator,
    water_fill_layers,
    apply_spans,
)
from parallax_amd.scheduling.model_info import ModelInfo
from parallax_amd.scheduling.node import MI355X, Node, NodeHardware
from parallax_amd.scheduling.scheduler import ClusterScheduler


def llama70b_info():
    cfg = ModelConfig(
        vocab_size=128256, hidden_size=8192, num_layers=80, num_heads=64,
        num_kv_heads=8, head_dim=128, intermediate_size=28672,
    )
    return ModelInfo("llama-70b", cfg)


def small_gpu(frac=0.25, name="small"):
    return NodeHardware(name=name, memory_gb=288 * frac,
                        tflops_bf16=2500 * frac, memory_bandwidth_gbps=8000 * frac)


def build_node(nid, hw=None):
    return Node(node_id=nid, hardware=hw or MI355X)


def set_full_rtt(nodes, rtt=2.0):
    for a in nodes:
        for b in nodes:
            if a is not b:
                a.rtt_ms[b.node_id] = rtt


def test_water_filling_respects_capacity_and_power():
    model = llama70b_info()
    nodes = [build_node("big"), build_node("small", small_gpu(0.25))]
    set_full_rtt(nodes)
    spans = water_fill_layers(nodes, model, 80)
    assert spans is not None
    apply_spans(nodes, spans)
    total = sum(e - s for s, e in spans)
    assert total == 80
    # power-proportional: big node gets ~4x the layers of the quarter node
    assert (spans[0][1] - spans[0][0]) > (spans[1][1] - spans[1][0]) * 2
    # contiguity
    assert spans[0][0] == 0 and spans[1][0] == spans[0][1] and spans[1][1] == 80


def test_greedy_single_big_node_single_pipeline():
    model = llama70b_info()
    nodes = [build_node("n0")]
    pipes = GreedyLayerAllocator(model).allocate_from_standby(nodes)
    assert len(pipes) == 1
    assert pipes[0].covers(80)
    assert pipes[0].nodes[0].num_layers_hosted == 80


def test_greedy_builds_multiple_pipelines():
    model = llama70b_info()
    nodes = [build_node(f"n{i}") for i in range(4)]
    set_full_rtt(nodes)
    pipes = GreedyLayerAllocator(model).allocate_from_standby(nodes)
    # one MI355X fits the whole 70B shard comfortably -> 4 pipelines
    assert len(pipes) == 4
    for p in pipes:
        assert p.covers(80)


def test_greedy_heterogeneous_pipeline():
    model = llama70b_info()
    # each small node holds a fraction; together they cover the model
    nodes = [build_node(f"s{i}", small_gpu(0.25, f"small{i}")) for i in range(6)]
    set_full_rtt(nodes)
    pipes = GreedyLayerAllocator(model).allocate_from_standby(nodes)
    assert len(pipes) >= 1
    assert all(p.covers(80) for p in pipes)
    # multi-node pipeline
    assert len(pipes[0].nodes) > 1


def test_dp_allocator_covers():
    model = llama70b_info()
    nodes = [build_node(f"n{i}") for i in range(3)]
    set_full_rtt(nodes)
    pipes = DynamicProgrammingLayerAllocator(model).allocate_from_standby(nodes)
    assert pipes and all(p.covers(80) for p in pipes)


class FixedCapNode(Node):
    """Fake node with a pinned layer capacity (capacity formula bypassed so
    partition tests can state exact heterogeneous pools)."""

    def __init__(self, nid, cap, hw=None):
        super().__init__(node_id=nid, hardware=hw or MI355X)
        self._cap = cap

    def decoder_layer_capacity(self, model=None, is_first=False, is_last=False):
        return self._cap


def test_dp_allocator_finds_interleaved_partition():
    """A heterogeneous pool where greedy/round-robin grouping
    cannot form two pipelines but the memoized dp(i, open_residuals, finished)
    search can. Capacities (40,35,30,30,25,20) over 90 layers: the only
    2-pipeline partition is {40,30,20} + {35,30,25}; round-robin over the
    capacity-sorted pool yields {40,30,25}=95 / {35,30,20}=85 < 90 and fails."""
    model = llama70b_info()
    model.cfg.num_layers = 90
    caps = {"a40": 40, "b35": 35, "c30": 30, "d30": 30, "e25": 25, "f20": 20}
    nodes = [FixedCapNode(nid, c) for nid, c in caps.items()]
    set_full_rtt(nodes)

    # the round-robin grouping (the old heuristic) cannot build k=2
    ordered = sorted(nodes, key=lambda n: n.decoder_layer_capacity(model),
                     reverse=True)
    rr = [[], []]
    for i, n in enumerate(ordered):
        rr[i % 2].append(n)
    assert min(sum(n.decoder_layer_capacity(model) for n in g) for g in rr) < 90

    pipes = DynamicProgrammingLayerAllocator(model).allocate_from_standby(nodes)
    assert len(pipes) == 2, f"DP should find 2 pipelines, got {len(pipes)}"
    for p in pipes:
        assert p.covers(90)
    groups = [sorted(caps[nid] for nid in p.node_ids) for p in pipes]
    assert sorted(groups) == [[20, 30, 40], [25, 30, 35]]


def test_dp_allocator_min_stages_prefers_fewer_nodes():
    """With one huge node and several small ones, k=1 via the huge node alone
    is a 1-stage pipeline; the DP must not smear layers across extra stages
    when a node pool supports more replicas."""
    model = llama70b_info()
    big = FixedCapNode("big", 100)
    smalls = [FixedCapNode(f"s{i}", 45) for i in range(2)]
    nodes = [big] + smalls
    set_full_rtt(nodes)
    pipes = DynamicProgrammingLayerAllocator(model).allocate_from_standby(nodes)
    # 80 layers: {big} alone and {s0,s1} together -> k=2 beats k=1
    assert len(pipes) == 2
    sizes = sorted(len(p.nodes) for p in pipes)
    assert sizes == [1, 2]
    assert all(p.covers(80) for p in pipes)


def make_scheduler(n_nodes=2, **kw):
    model = llama70b_info()
    sched = ClusterScheduler(model, min_nodes_bootstrapping=n_nodes, **kw)
    nodes = [build_node(f"n{i}") for i in range(n_nodes)]
    set_full_rtt(nodes)
    for n in nodes:
        sched.node_join(n)
    return sched, nodes


def test_bootstrap_and_dispatch():
    sched, nodes = make_scheduler(2)
    assert sched.bootstrapped
    d = sched.dispatch_next_request()
    assert d is not None
    table = d.routing_table
    # path is a registered, layer-covering pipeline
    assert table in [p.node_ids for p in sched.pipelines]
    assert all(sched.nodes[nid].current_requests == 1 for nid in table)
    sched.complete_request(table)
    assert all(sched.nodes[nid].current_requests == 0 for nid in table)


def test_round_robin_across_pipelines():
    sched, _ = make_scheduler(4)
    assert len(sched.pipelines) == 4
    seen = set()
    for _ in range(4):
        d = sched.dispatch_next_request()
        seen.add(tuple(d.routing_table))
        sched.complete_request(d.routing_table)
    assert len(seen) == 4  # round-robin touched every pipeline


def test_dynamic_join_after_bootstrap():
    model = llama70b_info()
    sched = ClusterScheduler(model, min_nodes_bootstrapping=1)
    first = build_node("first")
    sched.node_join(first)
    assert sched.bootstrapped
    # a quarter-size node joins: placed onto the lightest layers + rebalance
    late = build_node("late", small_gpu(0.25))
    late.rtt_ms["first"] = 2.0
    first.rtt_ms["late"] = 2.0
    assignment = sched.node_join(late)
    assert assignment is not None and assignment.end_layer > assignment.start_layer
    # pipeline still covers the model
    assert all(p.covers(80) for p in sched.pipelines)


def test_node_leave_rebalances_survivors():
    model = llama70b_info()
    sched = ClusterScheduler(model, min_nodes_bootstrapping=2)
    a, b = build_node("a"), build_node("b")
    set_full_rtt([a, b])
    sched.node_join(a)
    sched.node_join(b)
    assert sched.bootstrapped
    # two MI355X -> likely 2 pipelines; kill one node
    sched.node_leave("a")
    assert "a" not in sched.nodes
    # remaining pipelines (if any) still cover the model
    for p in sched.pipelines:
        assert p.covers(80)


def test_heartbeat_expiry():
    sched, nodes = make_scheduler(2)
    nodes[0].last_heartbeat -= 100.0
    expired = sched.sweep_heartbeats()
    assert nodes[0].node_id in expired
    assert nodes[0].node_id not in sched.nodes


def test_weight_refit_gate():
    sched, nodes = make_scheduler(1)
    sched.update_last_refit_time()
    # nodes report stale weights -> no eligible pipeline
    assert sched.dispatch_next_request() is None
    for n in nodes:
        n.last_refit_time = sched.last_refit_time
    assert sched.dispatch_next_request() is not None


def test_overload_gate():
    sched, nodes = make_scheduler(1)
    cap = nodes[0].max_requests(sched.model)
    nodes[0].current_requests = cap
    assert sched.dispatch_next_request() is None


def test_latency_routing_prefers_fast_pipeline():
    model = llama70b_info()
    sched = ClusterScheduler(model, min_nodes_bootstrapping=2,
                             routing_strategy="latency")
    fast = build_node("fast")
    slow = build_node("slow")
    set_full_rtt([fast, slow])
    sched.node_join(fast)
    sched.node_join(slow)
    slow.set_layer_latency_ms(50.0)
    fast.set_layer_latency_ms(1.0)
    d = sched.dispatch_next_request()
    assert d.routing_table == ["fast"]


def test_roofline_latency_sane():
    model = llama70b_info()
    n = build_node("n")
    n.start_layer, n.end_layer = 0, 80
    n.model = model
    lat = n.node_latency_ms(model)
    # 70B decode on one MI355X: ~>1 ms, < 1 s
    assert 0.5 < lat < 1000.0


def test_dijkstra_route_min_hop():
    from parallax_amd.scheduling.request_routing import dijkstra_route

    ranges = {
        "a": (0, 16), "b": (16, 32), "c": (0, 32),
        "d": (0, 8), "e": (8, 32),
    }
    # single node covering everything wins (1 hop)
    assert dijkstra_route(ranges, 32) == ["c"]
    # without c: 2-hop chains; either (a,b) or (d,e)
    del ranges["c"]
    path = dijkstra_route(ranges, 32)
    assert path in (["a", "b"], ["d", "e"])
    # unreachable coverage
    assert dijkstra_route({"a": (0, 16), "b": (20, 32)}, 32) is None


def test_dijkstra_route_latency_weighted():
    from parallax_amd.scheduling.request_routing import dijkstra_route

    ranges = {"a": (0, 16), "b": (16, 32), "d": (0, 16), "e": (16, 32)}
    lat = {("a", "b"): 10.0, ("a", "e"): 0.1, ("d", "e"): 10.0, ("d", "b"): 10.0}
    assert dijkstra_route(ranges, 32, latency=lat) == ["a", "e"]


def test_dp_allocator_prefers_parallel_pipelines():
    """Z(k) = k^2/(T + stages/k * RTT): with 4 over-half-capacity nodes the
    DP allocator should build 2 two-stage pipelines (throughput 4) rather
    than one four-stage chain (reference DP objective,
    layer_allocation.py:758+)."""
    model = llama70b_info()
    nodes = [build_node(f"n{i}", small_gpu(0.6, f"half{i}")) for i in range(4)]
    set_full_rtt(nodes, rtt=2.0)
    pipelines = DynamicProgrammingLayerAllocator(model).allocate_from_standby(nodes)
    assert pipelines and len(pipelines) == 2
    for p in pipelines:
        assert p.covers(80)
        spans = sorted((n.start_layer, n.end_layer) for n in p.nodes)
        for (s0, e0), (s1, e1) in zip(spans, spans[1:]):
            assert e0 == s1  # contiguous coverage


def test_greedy_lookahead_closes_with_smallest_node():
    """Greedy look-ahead: when a pipeline needs a closer, pick the SMALLEST
    node able to close it so big nodes seed the next pipeline
    (layer_allocation.py:582-755 behavior)."""
    model = llama70b_info()
    nodes = [
        build_node("big0", small_gpu(0.55, "b0")),   # ~64-layer capacity
        build_node("big1", small_gpu(0.55, "b1")),
        build_node("small0", small_gpu(0.25, "s0")), # ~29-layer capacity
        build_node("small1", small_gpu(0.25, "s1")),
    ]
    set_full_rtt(nodes)
    pipelines = GreedyLayerAllocator(model).allocate_from_standby(nodes)
    assert len(pipelines) == 2
    for p in pipelines:
        ids = {n.node_id for n in p.nodes}
        # each pipeline pairs one big with one small — big nodes are not
        # burned as closers for each other
        assert len(ids & {"big0", "big1"}) == 1
        assert len(ids & {"small0", "small1"}) == 1


def test_allocation_fails_cleanly_when_undercapacity():
    model = llama70b_info()
    nodes = [build_node("tiny", small_gpu(0.05, "t"))]
    set_full_rtt(nodes)
    assert GreedyLayerAllocator(model).allocate_from_standby(nodes) == []
    assert water_fill_layers(nodes, model, 80) is None


def test_detect_hardware_cpu_profile():
    from parallax_amd.scheduling.node import detect_hardware

    hw = detect_hardware()
    assert hw.memory_gb > 0 and hw.tflops_bf16 > 0
    n = Node(node_id="d", hardware=hw)
    assert n.decoder_layer_capacity(llama70b_info()) >= 0


try:
    from hypothesis import HealthCheck, given, settings
    from hypothesis import strategies as st
    HAVE_HYP = True
except ImportError:  # pragma: no cover
    HAVE_HYP = False


@pytest.mark.skipif(not HAVE_HYP, reason="hypothesis not installed")
@settings(max_examples=40, deadline=None,
          suppress_health_check=[HealthCheck.too_slow])
@given(fracs=st.lists(st.sampled_from([0.15, 0.25, 0.5, 1.0]),
                      min_size=1, max_size=6),
       algo=st.sampled_from(["greedy", "dp"]))
def test_allocators_structural_invariants(fracs, algo):
    """For ANY node mix, every produced pipeline must cover [0, L)
    contiguously with disjoint spans, respect each node's layer capacity,
    and never reuse a node across pipelines."""
    model = llama70b_info()
    nodes = [build_node(f"n{i}", small_gpu(f, name=f"hw{i}"))
             for i, f in enumerate(fracs)]
    set_full_rtt(nodes)
    cls = (GreedyLayerAllocator if algo == "greedy"
           else DynamicProgrammingLayerAllocator)
    pipelines = cls(model).allocate_from_standby(list(nodes))
    L = model.num_layers
    used = set()
    for pipe in pipelines:
        spans = [(n.start_layer, n.end_layer) for n in pipe.nodes]
        # contiguous cover of [0, L)
        assert spans[0][0] == 0 and spans[-1][1] == L
        for (s0, e0), (s1, e1) in zip(spans, spans[1:]):
            assert e0 == s1 and e0 > s0
        assert all(e > s for s, e in spans)
        for n in pipe.nodes:
            assert n.node_id not in used, "node reused across pipelines"
            used.add(n.node_id)
            cap = n.decoder_layer_capacity(model)
            assert n.end_layer - n.start_layer <= cap


@pytest.mark.skipif(not HAVE_HYP, reason="hypothesis not installed")
@settings(max_examples=25, deadline=None,
          suppress_health_check=[HealthCheck.too_slow])
@given(fracs=st.lists(st.sampled_from([0.12, 0.2, 0.3, 0.5]),
                      min_size=2, max_size=5))
def test_dp_minimum_stages_vs_bruteforce(fracs):
    """For every feasible pipeline count k, the DP's chosen partition must
    use no more total stages than ANY brute-force partition of the pool
    into k feasible pipelines (exhaustive set-partition check, N<=5)."""
    from itertools import combinations

    model = llama70b_info()
    nodes = [build_node(f"b{i}", small_gpu(f, name=f"b{i}"))
             for i, f in enumerate(fracs)]
    set_full_rtt(nodes)
    L = model.num_layers
    caps = {n.node_id: n.decoder_layer_capacity(model) for n in nodes}

    def feasible(group):
        # position-aware: the first node also hosts the embedding and the
        # last the lm_head, shrinking their layer capacity — pick the
        # best (first, last) assignment for the group
        if len(group) == 1:
            n = group[0]
            return n.decoder_layer_capacity(
                model, is_first=True, is_last=True) >= L
        best = -1
        for f in group:
            for last in group:
                if f is last:
                    continue
                tot = sum(
                    n.decoder_layer_capacity(
                        model, is_first=(n is f), is_last=(n is last))
                    for n in group
                )
                best = max(best, tot)
        return best >= L

    def best_bruteforce(k):
        """Min total nodes used across partitions into k feasible groups."""
        ids = list(range(len(nodes)))

        def rec(remaining, k_left):
            if k_left == 0:
                return 0
            if len(remaining) < k_left:
                return None
            best = None
            # first group: any subset containing remaining[0]... also allow
            # leaving nodes unused: choose subsets of remaining
            head = remaining[0]
            rest = remaining[1:]
            # option: head unused
            r = rec(rest, k_left)
            if r is not None:
                best = r
            for sz in range(1, len(rest) + 2):
                for combo in combinations(rest, sz - 1):
                    group = [nodes[head]] + [nodes[c] for c in combo]
                    if not feasible(group):
                        continue
                    rem2 = [x for x in rest if x not in combo]
                    r = rec(rem2, k_left - 1)
                    if r is not None:
                        tot = sz + r
                        if best is None or tot < best:
                            best = tot
            return best

        return rec(ids, k)

    alloc = DynamicProgrammingLayerAllocator(model)
    pipes = alloc.allocate_from_standby(list(nodes))
    if not pipes:
        # DP says infeasible for every k: brute force must agree for k=1
        assert best_bruteforce(1) is None
        return
    k = len(pipes)
    dp_stages = sum(len(p.nodes) for p in pipes)
    bf = best_bruteforce(k)
    assert bf is not None
    assert dp_stages <= bf, (dp_stages, bf, fracs, k)
