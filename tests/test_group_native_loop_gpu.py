"""TP groups on the native serving loop (runtime/mirror.h): the leader's C++ EngineLoop
serves the requests and its followers' EngineMirror threads replay its device operations
-- prefill chunks and (multi-step) decode graphs with their IPC collectives -- with no
Python on the hot path of any rank.  Ranks are virtual (every rank process on the one GPU
of the test box, IPC collectives between the processes), the group is a real
ClusterServer replica.

Replies must equal the same group's Python lockstep loop (ENGINE_NATIVE_LOOP=0: the
round-4 path, pickled plans over the pipes) -- greedy and seeded sampling, riders and
concurrent requests -- and the leader's metrics must show the mirror at work.  (The
reference serves one click per Ollama call, `web/streamlit_app.py:161-173`; BASELINE
configs 3 and 5 serve it from TP / EP groups.)"""
import json
import os
import threading

import pytest

from p2p_llm_chat_go_amd.engine.cluster import ClusterServer

pytestmark = pytest.mark.gpu

MSGS = ["Did you see the game last night? That last-minute goal was unbelievable!",
        "Hey! How's it going?", "Are we still on for lunch tomorrow at noon?",
        "Quick question: do you know where the spare keys for the storage room are?"]


def _req(i, sampled=False, n=24):
    opts = {"num_predict": n, "ignore_eos": True}
    if sampled:
        opts.update(temperature=0.8, top_k=40, top_p=0.9, seed=100 + i)
    return json.dumps({"model": "llama3.1", "prompt": MSGS[i % len(MSGS)], "stream": False,
                       "options": opts})


def _serve(world, native, reqs):
    env = {"ENGINE_NATIVE_LOOP": "1" if native else "0", "P2P_CAR_TIMEOUT_MS": "30000",
           "P2P_QA_TIMEOUT_MS": "30000",
           # the fused all-reduce epilogue at every width: its launch keeps to the ranks'
           # share of the one device (tests/test_world8_gpu.py explains the residency limit)
           "P2P_TP_FUSED_AR": os.environ.get("P2P_TP_FUSED_AR", "1")}
    old = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    try:
        cs = ClusterServer("tiny-llama-gqa", gpus=world, tp=world, device="cuda", sd_seed=3,
                           max_batch=2, warmup=False, virtual_ranks=True, start_timeout=600,
                           kv_pages=256)
    finally:
        for k, v in old.items():
            if v is None:
                os.environ.pop(k, None)
            else:
                os.environ[k] = v
    try:
        seq = [json.loads(cs.handle_json(r)) for r in reqs]  # one at a time
        conc = [None] * len(reqs)

        def run(i):
            conc[i] = json.loads(cs.handle_json(reqs[i]))

        ths = [threading.Thread(target=run, args=(i,)) for i in range(len(reqs))]
        [t.start() for t in ths]
        [t.join(timeout=300) for t in ths]
        # a full batch (max_batch = 2) of long replies with nobody waiting: 8-step chunks
        full = [None] * 2
        ths = [threading.Thread(target=lambda i=i: full.__setitem__(
            i, json.loads(cs.handle_json(_req(i, n=96))))) for i in range(2)]
        [t.start() for t in ths]
        [t.join(timeout=300) for t in ths]
        assert all(f is not None and f["eval_count"] == 96 for f in full)
        m = cs.metrics()
    finally:
        cs.close()
    return seq, conc, m


@pytest.mark.parametrize("world", [2, 4, 8])
def test_group_native_loop_matches_python_lockstep(world):
    reqs = [_req(0), _req(1), _req(2, sampled=True), _req(3, n=40)]
    seq_n, conc_n, m = _serve(world, True, reqs)
    rep = m["per_replica"][0]
    assert rep.get("native_loop") == 1 and rep.get("mirror_frames", 0) > 0, rep
    show = {k: rep.get(k) for k in ("k_step_graphs", "k_graph_launches", "decode_calls",
                                     "decode_steps", "captures", "prefill_calls",
                                     "eager_prefill_calls", "mirror_frames")}
    assert rep.get("k_step_graphs", 0) > 0, show  # captured collectively on every rank
    assert rep.get("k_graph_launches", 0) > 0, show  # and replayed as whole k-step graphs
    seq_p, _conc_p, mp = _serve(world, False, reqs)
    assert "mirror_frames" not in mp["per_replica"][0]
    # every reply in full, the seeded sampled one (request 2) included: both loops run a
    # chunk shape eagerly until its n-th use and through its captured graph after, and the
    # two forms' logits are pinned directly by test_tp_prefill_graph_matches_eager below
    # (bit-identical at 2 / 4 / 8 ranks)
    for i, (a, b) in enumerate(zip(seq_n, seq_p)):
        assert a["eval_count"] == b["eval_count"]
        assert a["response"] == b["response"], (i, a["response"], b["response"])
    # concurrent (batched decode, riders in prompt chunks): every reply complete (the
    # batch shapes differ from the sequential run's, so bf16 rounding may flip near-ties)
    for a, b in zip(conc_n, seq_p):
        assert a is not None and a["done"] and a["eval_count"] == b["eval_count"]


def test_group_follower_fault_fails_the_step():
    """a kernel fault is local to the rank that saw it.  A follower whose split-K
    fault word is set (P2P_MIRROR_INJECT_FAULT: after its 3rd launching frame, inside the
    first request) reports it on the group channel's status back channel (runtime/mirror.h);
    the leader fails exactly that request with the reason, every rank's words are cleared,
    and the next request's reply equals a clean group's."""
    os.environ["P2P_MIRROR_INJECT_FAULT"] = "3"
    try:
        cs = ClusterServer("tiny-llama-gqa", gpus=2, tp=2, device="cuda", sd_seed=3, max_batch=2,
                           warmup=False, virtual_ranks=True, start_timeout=600, kv_pages=256)
    finally:
        os.environ.pop("P2P_MIRROR_INJECT_FAULT", None)
    try:
        with pytest.raises(RuntimeError, match="follower rank"):
            cs.handle_json(_req(0))
        after = json.loads(cs.handle_json(_req(0)))
        m = cs.metrics()["per_replica"][0]
    finally:
        cs.close()
    assert m.get("mirror_follower_faults", 0) >= 1, m
    clean, _conc, _m = _serve(2, True, [_req(0)])
    assert after["response"] == clean[0]["response"] and after["eval_count"] == 24


def test_group_follower_collective_timeout_kills_the_replica():
    """A collective timeout is not transient: the rank's later IPC calls skip their waits, so
    every sum after it is wrong.  A follower whose collectives' timeout word is set
    (P2P_MIRROR_INJECT_COLL: after its 3rd launching frame) reports it as its own status bit;
    the leader fails the request with the reason and marks the replica dead, and the router
    refuses the next request instead of serving it from a broken group."""
    import time

    os.environ["P2P_MIRROR_INJECT_COLL"] = "3"
    try:
        cs = ClusterServer("tiny-llama-gqa", gpus=2, tp=2, device="cuda", sd_seed=3, max_batch=2,
                           warmup=False, virtual_ranks=True, start_timeout=600, kv_pages=256)
    finally:
        os.environ.pop("P2P_MIRROR_INJECT_COLL", None)
    try:
        with pytest.raises(RuntimeError, match="collective timeout"):
            cs.handle_json(_req(0))
        time.sleep(2.0)  # the replica's watchdog reports the dead loop
        with pytest.raises(RuntimeError):
            cs.handle_json(_req(1))
    finally:
        cs.close()


def _port():
    import socket

    s = socket.socket()
    s.bind(("127.0.0.1", 0))
    p = s.getsockname()[1]
    s.close()
    return p


def _forms_worker(rank, world, port, q):
    """One TP rank: every chat prompt's chunk through the eager prefill and through its
    captured prefill graph (sampled form: fp32 logits + the vocab-parallel draw), twice each."""
    import torch
    import torch.distributed as dist

    os.environ.update(MASTER_ADDR="127.0.0.1", MASTER_PORT=str(port), P2P_CAR_TIMEOUT_MS="30000",
                      P2P_QA_TIMEOUT_MS="30000")
    dist.init_process_group("gloo", rank=rank, world_size=world)
    eng = None
    try:
        from p2p_llm_chat_go_amd.engine import Engine
        from p2p_llm_chat_go_amd.engine.kv_cache import pages_for
        from p2p_llm_chat_go_amd.engine.sampling import SamplingParams
        from p2p_llm_chat_go_amd.models.config import TINY_LLAMA_GQA
        from p2p_llm_chat_go_amd.models.reference import random_state_dict
        from p2p_llm_chat_go_amd.models.weights import EngineWeights
        from p2p_llm_chat_go_amd.parallel.comm import TPComm

        torch.cuda.set_device(0)
        cfg = TINY_LLAMA_GQA
        sd = random_state_dict(cfg, seed=3, device="cuda", on_device=True)
        w = EngineWeights.from_state_dict(sd, cfg, "cuda", tp_rank=rank, tp_size=world)
        eng = Engine(cfg, weights=w, device="cuda", kv_pages=64, max_batch=2, comm=TPComm(),
                     tp_rank=rank, tp_size=world, use_graph=True)
        out = []
        for n, L in enumerate((14, 23, 37, 44)):
            p = [(101 + 37 * i + 13 * n) % (cfg.vocab - 10) + 5 for i in range(L)]
            sp = SamplingParams(temperature=0.8, top_k=40, top_p=0.9, seed=100 + n)
            pages = eng.kv.allocator.alloc(pages_for(L + 8))
            res = {}
            for form in ("eager", "graph"):
                for rep in range(2):
                    if form == "eager":
                        f, lg = eng.prefill([p], [pages], return_logits=True, sampling=[sp],
                                            graph=False)
                        lg = lg[:1]
                    else:
                        rows = [(0, i, t) for i, t in enumerate(p)]
                        f = eng._prefill_graphed([p], [pages], rows, L, [sp], True)
                        lg = eng.prefill_graph(L, 1, L, greedy=False).ws.logits[:1]
                    lg = lg.float().cpu().clone()
                    parts = [torch.empty_like(lg) for _ in range(world)]
                    dist.all_gather(parts, lg)
                    # numpy: pickled by value (a tensor in the queue is a shared-memory handle
                    # that dies with this process)
                    res[form, rep] = (int(f[0].item()), torch.cat(parts, 1).numpy())
            eng.kv.allocator.free(pages)
            eng.check_comm()
            out.append((L, res))
        q.put((rank, True, out if rank == 0 else None))
    except Exception:
        import traceback

        q.put((rank, False, traceback.format_exc()))
    finally:
        try:
            eng.model.comm.close()
        except Exception:
            pass
        dist.destroy_process_group()


@pytest.mark.parametrize("world", [2, 4, 8])
def test_tp_prefill_graph_matches_eager(world):
    """the direct check behind the sampled-reply comparison above.  A TP
    prompt chunk run eagerly and through its captured prefill graph (IPC collectives inside
    the graph, prompt rows padded to the row bucket) gives the same vocab-sharded logits up
    to bf16 rounding, each form is bit-reproducible run to run, and wherever the two forms'
    logits are bit-identical they draw the same seeded first token."""
    import multiprocessing as mp

    import numpy as np

    ctx = mp.get_context("spawn")
    q = ctx.Queue()
    port = _port()
    ps = [ctx.Process(target=_forms_worker, args=(r, world, port, q)) for r in range(world)]
    [p.start() for p in ps]
    res = []
    try:
        for _ in range(world):
            res.append(q.get(timeout=300))
    finally:
        [p.join(timeout=30) for p in ps]
        [p.terminate() for p in ps if p.is_alive()]
    for rank, ok, info in sorted(res, key=lambda r: r[0]):
        assert ok, (rank, info)
    out = [info for rank, _, info in res if rank == 0][0]
    report = []
    for L, r in out:
        (fe, le), (fe2, le2) = r["eager", 0], r["eager", 1]
        (fg, lg), (fg2, lg2) = r["graph", 0], r["graph", 1]
        assert np.array_equal(le, le2) and fe == fe2, ("eager prefill not reproducible", L)
        assert np.array_equal(lg, lg2) and fg == fg2, ("graph prefill not reproducible", L)
        d = float(np.abs(le - lg).max())
        spread = float(le.std())
        report.append((L, d, spread, fe, fg))
        assert d <= 0.02 * spread + 1e-3, ("graph vs eager logits", L, d, spread)
        if d == 0.0:
            assert fe == fg, ("bit-identical logits drew different tokens", L, fe, fg)
    print("world %d: (prompt rows, max |graph - eager|, logit std, eager tok, graph tok) %s"
          % (world, report))



def _serve_a2a(native, reqs, world=4):
    env = {"ENGINE_NATIVE_LOOP": "1" if native else "0", "P2P_CAR_TIMEOUT_MS": "30000",
           "P2P_QA_TIMEOUT_MS": "30000"}
    old = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    try:
        cs = ClusterServer("tiny-mixtral-8e", gpus=world, ep=world, device="cuda", sd_seed=3,
                           max_batch=4, warmup=False, virtual_ranks=True, start_timeout=600,
                           kv_pages=256, ep_mode="a2a")
    finally:
        for k, v in old.items():
            if v is None:
                os.environ.pop(k, None)
            else:
                os.environ[k] = v
    try:
        seq = [json.loads(cs.handle_json(r)) for r in reqs]
        conc = [None] * len(reqs)

        def run(i):
            conc[i] = json.loads(cs.handle_json(reqs[i]))

        ths = [threading.Thread(target=run, args=(i,)) for i in range(len(reqs))]
        [t.start() for t in ths]
        [t.join(timeout=300) for t in ths]
        m = cs.metrics()
    finally:
        cs.close()
    return seq, conc, m


def test_ep_a2a_group_on_native_loop_matches_python_lockstep():
    """the EP all-to-all mode (DP attention: every sequence lives on one
    rank, experts exchanged with all-to-all) on the native loop.  The leader's EngineLoop
    gives each new sequence a home rank, runs every rank's share through the same shapes
    (prefill padded to the largest share, decode at the largest share's batch bucket), each
    follower's frame carries its own share's metadata, and its tokens come back with the
    frame's status (runtime/mirror.h 'T' / 'E' records).  Replies -- greedy and seeded
    sampled, one at a time and concurrent (several ranks busy at once) -- equal the Python
    lockstep loop's (engine/cluster.py LockstepEngine dp_split), and the metrics show the
    native loop and its mirror frames at work."""
    reqs = [_req(0), _req(1), _req(2, sampled=True), _req(3, n=40), _req(1, n=16)]
    seq_n, conc_n, m = _serve_a2a(True, reqs)
    rep = m["per_replica"][0]
    assert rep.get("native_loop") == 1 and rep.get("mirror_frames", 0) > 0, rep
    assert rep.get("dp_world") == 4 and rep.get("eager_prefill_calls", 0) > 0, rep
    seq_p, conc_p, mp = _serve_a2a(False, reqs)
    assert "mirror_frames" not in mp["per_replica"][0]
    for i, (a, b) in enumerate(zip(seq_n, seq_p)):
        assert a["eval_count"] == b["eval_count"], (i, a, b)
        assert a["response"] == b["response"], (i, a["response"], b["response"])
    # concurrent: the shares differ from the sequential run's (other ranks, other batch
    # buckets), so only completeness is compared
    for a, b in zip(conc_n, seq_p):
        assert a is not None and a["done"] and a["eval_count"] == b["eval_count"]
