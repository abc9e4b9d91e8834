"""Performance cases of the batched Hive engine, through its public entry points.

Each case is one call (or one short fixed sequence of calls) that a program of
this framework makes in earnest: the legal lists, features and action indices
of a batch of positions, whole random games, the training forward batch, the
leaf evaluation of a search wave, the root tactical probe, and whole self-play
plies.  Positions come from the engine's seeded random play, as the
benchmark's do.

A case's `kind` says which call it is:

  lists   generate_legal_moves_features_actions_batch: the fused encoder pass
  pair    generate_legal_moves_and_fnn_features_batch, then
          legal_moves_to_actions_batch: the reference's own two calls
  play    random_positions in lockstep: whole random games
  train   build_forward_batch: root features and every legal successor's
  leaf    fnn_leaf_eval_lists: priors, values and child Q of a wave's leaves
  probe   root_tactical_probe_batch with every stage on
  search  one self-play ply: search_ply, then apply_and_rebase
"""
import math

import numpy as np
import torch

from hive_neuralnet_amd import hive_gpu
from hive_neuralnet_amd.fnn import seeded_large
from hive_neuralnet_amd.orchestrator import FNNMCTSConfig, FNNMCTSOrchestrator
from hive_neuralnet_amd.replay import build_forward_batch

STATE, MOVES, FEAT, ACTIONS = 3424, 256 * 6, 122 * 4, 256 * 4  # bytes of a row
ROW_FLOPS = 2 * (122 * 64 + 64 * 64 + 64 * 64 + 64 + 64)  # one feature row through the 64-wide network


def listed():
    return [
        # one position with every expansion piece: a GUI's or an analysis tool's call, all latency
        {"name": "lists_one", "kind": "lists", "batch": 1, "mask": 7, "max_ply": 60},
        # the benchmark's headline batch: base game, 65,536 positions
        {"name": "lists_base", "kind": "lists", "batch": 65536, "mask": 0, "max_ply": 120},
        # the same batch with mosquito, ladybug and pillbug
        {"name": "lists_expansion", "kind": "lists", "batch": 65536, "mask": 7, "max_ply": 150},
        # a data set's ragged remainder through the reference's two calls
        {"name": "pair_ragged", "kind": "pair", "batch": 2999, "mask": 7, "max_ply": 100},
        # 16,384 whole random games: the lockstep benchmark
        {"name": "play_games", "kind": "play", "batch": 16384, "mask": 0, "max_ply": 300},
        # the trainer's forward batch, legal lists generated
        {"name": "train_batch", "kind": "train", "batch": 2048, "mask": 0, "max_ply": 120, "cached": False},
        # the leaves of one mid-game self-play wave at 512 games and 16 candidates
        {"name": "leaf_wave", "kind": "leaf", "batch": 8192, "mask": 0, "max_ply": 120},
        # the leaves of a wave of a few games
        {"name": "leaf_few", "kind": "leaf", "batch": 77, "mask": 7, "max_ply": 60},
        # the trainer's default root analysis over the benchmark's batch
        {"name": "probe_roots", "kind": "probe", "batch": 4096, "mask": 0, "max_ply": 150},
        # one ply of the self-play benchmark, mid-game: 512 games, 4,096 simulations a move
        {"name": "search_selfplay", "kind": "search", "batch": 512, "mask": 0, "max_ply": 120, "sims": 4096,
         "waves": True},
        # one ply from the empty board with one simulation per candidate per wave
        {"name": "search_single", "kind": "search", "batch": 128, "mask": 0, "max_ply": 0, "sims": 1024,
         "waves": False},
        # one ply of a few games at the configuration's default 128 simulations
        {"name": "search_few", "kind": "search", "batch": 16, "mask": 7, "max_ply": 60, "sims": 128, "waves": True},
    ]


def draw(rng):
    def size(lo, hi):  # spread over the logarithm, odd sizes among them
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["lists", "lists", "pair", "play", "train", "leaf", "leaf", "probe", "search", "search"])
    case = {"kind": kind, "mask": rng.choice([0, 0, 7, rng.randrange(8)]), "max_ply": rng.randrange(20, 151)}
    if kind in ("lists", "pair"):
        case["batch"] = size(1, 65536)
    elif kind == "play":
        case["batch"] = size(32, 8192)
        case["max_ply"] = rng.randrange(20, 301)
    elif kind == "train":
        case["batch"] = size(16, 2048)
        case["cached"] = rng.random() < 0.5
    elif kind == "leaf":
        case["batch"] = size(8, 8192)
    elif kind == "probe":
        case["batch"] = size(8, 4096)
    else:
        case["batch"] = size(4, 256)
        case["sims"] = size(64, 1024)
        case["waves"] = rng.random() < 0.7
    return case


class State:
    """What a program holds before the call."""


def _train_positions(ext, case, seed):
    """Positions whose legal moves add up to the case's row count, so that
    every batch of a case has the same number of successor rows."""
    B = case["batch"]
    pool = hive_gpu.random_positions(3 * B + 64, case["mask"], case["max_ply"], seed)[0]
    n = ext.generate_legal_moves_batch(pool, pool.shape[0])[1].cpu().numpy().astype(np.int64)
    take, spare = np.arange(B), np.arange(B, pool.shape[0])
    for _ in range(1000):  # exchange one position for another until the sum is met
        short = int(B * _legal(case)) - int(n[take].sum())
        if short == 0:
            break
        i = int(np.argmin(n[take]) if short > 0 else np.argmax(n[take]))
        j = int(np.argmin(np.abs(n[spare] - n[take[i]] - short)))
        take[i], spare[j] = spare[j], take[i]
    return pool[torch.from_numpy(take).cuda()].contiguous()


def prepare(case, seed):
    s = State()
    s.case, s.seed = case, int(seed)
    s.ext = hive_gpu.load_extension()
    B, kind = case["batch"], case["kind"]
    if kind == "play":
        return s
    if kind == "train":
        s.states = _train_positions(s.ext, case, s.seed)
    elif case["max_ply"] > 0:
        s.states = hive_gpu.random_positions(B, case["mask"], case["max_ply"], s.seed)[0]
    else:
        s.states = s.ext.create_initial_states(B, case["mask"])
    if kind == "train" and case["cached"]:  # the replay buffer's cached columns
        s.moves, n, feat = s.ext.generate_legal_moves_and_fnn_features_batch(s.states, B)
        s.num_legal, s.features = n.to(torch.int64), feat.to(torch.float16)
    elif kind == "leaf":
        s.moves, s.num_legal, s.features = s.ext.generate_legal_moves_and_fnn_features_batch(s.states, B)
        s.net = seeded_large(s.seed)
        s.biases = (float(s.net.value_fc.bias.item()), float(s.net.action_fc2.bias.item()))
        s.workspace = torch.empty((s.ext.leaf_eval_workspace_bytes(B),), dtype=torch.uint8, device="cuda")
    elif kind == "probe":
        s.moves, s.num_legal = s.ext.generate_legal_moves_batch(s.states, B)
        g = torch.Generator(device="cuda").manual_seed(s.seed)
        s.priors = torch.rand((B, 256), generator=g, device="cuda")
    elif kind == "search":
        cfg = FNNMCTSConfig(num_simulations=case["sims"], batch_size=B, expansion_mask=case["mask"],
                            wave_parallel=case["waves"], max_tree_nodes=1 + case["sims"] * 256)
        s.search = FNNMCTSOrchestrator(seeded_large(s.seed), cfg)
        s.tree = s.search._alloc_tree(B)
        s.active = s.ext.check_results_batch(s.states, B) == 0
        s.board = s.states.clone()
    return s


def run(s):
    case, B = s.case, s.case["batch"]
    kind = case["kind"]
    if kind == "lists":
        return s.ext.generate_legal_moves_features_actions_batch(s.states, B)
    if kind == "pair":
        moves, n, feat = s.ext.generate_legal_moves_and_fnn_features_batch(s.states, B)
        return moves, n, feat, s.ext.legal_moves_to_actions_batch(s.states, moves, n, B)
    if kind == "play":
        return hive_gpu.random_positions(B, case["mask"], case["max_ply"], s.seed, lockstep=True)
    if kind == "train":
        if case["cached"]:
            return build_forward_batch(s.ext, s.states, B, s.num_legal, s.features, s.moves)
        return build_forward_batch(s.ext, s.states, B)
    if kind == "leaf":
        return s.ext.fnn_leaf_eval_lists(s.states, s.moves, s.num_legal, s.features, B, s.net, s.biases, s.workspace)
    if kind == "probe":
        return s.ext.root_tactical_probe_batch(s.states, s.moves, s.num_legal, s.priors, B)
    # a ply from the same roots every time: the boards are put back, the trees
    # were reset by the last ply's rebase
    s.board.copy_(s.states)
    torch.manual_seed(s.seed)
    np.random.seed(s.seed & 0x7FFFFFFF)
    ply = s.search.search_ply(s.board, s.tree, s.active)
    s.search.apply_and_rebase(s.board, s.tree, ply)
    return {"policy": ply.policy, "visits": ply.slot_visits, "chosen": ply.chosen_slot, "legal": ply.legal_moves,
            "num_legal": ply.num_legal, "states": s.board}


def _legal(case):
    """Mean legal moves of a position, about: 52 in the base game, 6 more for
    each expansion piece, fewer when the play ends early."""
    if case["max_ply"] == 0:
        return 20
    return (52 + 6.3 * bin(case["mask"]).count("1")) * min(1.0, 0.58 + 0.006 * case["max_ply"])


def work(case):
    B, L, kind = case["batch"], _legal(case), case["kind"]
    if kind in ("lists", "pair"):
        return {"bytes": B * (STATE + MOVES + 4 + FEAT + ACTIONS), "flops": 0}
    if kind == "play":
        return {"bytes": B * (STATE + 4), "flops": 0}
    if kind == "train":
        return {"bytes": B * (STATE + FEAT + 8 + L * (6 + FEAT + 8)), "flops": 0}
    if kind == "leaf":
        return {"bytes": B * (STATE + 4 + FEAT + 6 * L + 2 * 1024 + 4), "flops": B * (1 + L) * ROW_FLOPS}
    if kind == "probe":
        return {"bytes": B * (STATE + MOVES + 4 + 1024 + 8 + 256 + 1), "flops": 0}
    # per simulation: a leaf row read, its legal list, the priors and child Q of its children; in and out of the tree
    sims = B * case["sims"]
    return {"bytes": sims * (STATE + L * (6 + 8 + 47)), "flops": sims * (1 + L) * ROW_FLOPS}


def tolerance(case):
    if case["kind"] == "leaf":  # float32 sums of 64 to 122 terms
        return {"rel": 1e-5, "max": 1e-4}
    if case["kind"] == "search":
        # network outputs that differ by one part in 1e7 change a few of a game's simulations: policies were
        # 1e-6 to 2e-3 apart (512 games), visits and chosen moves the same
        return {"rel": 1e-2, "max": 0.9, "differ": 0.005}
    return "exact"


def exact(case, seed):
    """The network of the `leaf` cases in 64 bits over the engine's feature
    rows (quotients of small whole numbers, inputs here); the other kinds'
    outputs are whole numbers and such quotients, or follow from a whole search."""
    if case["kind"] != "leaf":
        return None
    s = prepare(case, seed)
    B = case["batch"]
    n = s.num_legal.to(torch.int64)
    slot = torch.arange(256, device="cuda").unsqueeze(0).expand(B, -1)
    valid = slot < n.unsqueeze(1)
    root = torch.arange(B, device="cuda").unsqueeze(1).expand(-1, 256)[valid]
    rows = s.ext.fnn_successor_features_batch(s.states, s.moves, root, slot[valid], int(root.shape[0])).double()
    w = {k: v.detach().double() for k, v in s.net.state_dict().items()}

    def linear(x, name):
        return x @ w[name + ".weight"].t() + w[name + ".bias"]

    def encode(x):
        h = torch.sigmoid(linear(x, "fc1"))
        h = h - h.mean(dim=1, keepdim=True)
        h = h / torch.sqrt((h * h).mean(dim=1, keepdim=True) + 1e-5)
        return linear(h * w["ln1.weight"] + w["ln1.bias"], "fc2")

    e0 = encode(s.features.double())
    half = w["action_fc1.weight"]
    logits = torch.full((B, 256), -math.inf, dtype=torch.float64, device="cuda")
    child_q = torch.zeros((B, 256), dtype=torch.float64, device="cuda")
    flat_logit, flat_value = [], []
    root_half = e0 @ half[:, :64].t() + w["action_fc1.bias"]
    for at in range(0, rows.shape[0], 1 << 16):
        e = encode(rows[at: at + (1 << 16)])
        flat_value.append(torch.tanh(linear(e, "value_fc")).squeeze(1))
        h = torch.sigmoid(root_half[root[at: at + (1 << 16)]] + e @ half[:, 64:].t())
        flat_logit.append(linear(h, "action_fc2").squeeze(1))
    if flat_logit:
        logits[valid] = torch.cat(flat_logit)
        child_q[valid] = -torch.cat(flat_value)
    priors = torch.nan_to_num(torch.softmax(logits, dim=1), nan=0.0)
    return priors, torch.tanh(linear(e0, "value_fc")).squeeze(1), child_q
