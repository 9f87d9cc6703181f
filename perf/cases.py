"""The work this framework is used for, as cases that can be timed.

Every case goes through the public Python surface (chessrl_amd.models): leaf evaluation with the
BT4-class encoder, move prediction, scoring and rollouts with the GPT model, loss evaluation and
1-ply search with BT4. Models are full size, built once per process and shared by the batches that
go through them, as a search or training loop keeps one model and feeds it new positions; positions
are seeded random playouts.
"""
import torch

from chessrl_amd import board, models

VOCAB_RL, VOCAB_LEELA = models.VOCAB_RL, models.VOCAB_LEELA
DEV = "cuda"
GPT_LAYERS, GPT_HEADS, GPT_C, GPT_BLOCK = 6, 12, 768, 256       # GPTConfig's defaults, the reference's block size
BT4_L, BT4_C, BT4_F = 10, 512, 736                              # BT4's defaults
LEAF_L, LEAF_C, LEAF_F, LEAF_H = 15, 1024, 1536, 32             # the benchmark encoder
CHILDREN = 31                                                    # mean legal moves of a playout position
MOST_MOVES = 218                                                 # most legal moves of any position
START_THINK, END_THINK, END_VARIATION, END = 1924, 1925, 1926, 1927


def listed():
    return [
        # One leaf of a tree search that waits for its answer: nothing but latency.
        {"name": "leaf_bf16_b1", "kind": "leaf", "dtype": "bf16", "batch": 1},
        # The batch of leaves a parallel tree search collects.
        {"name": "leaf_bf16_b64", "kind": "leaf", "dtype": "bf16", "batch": 64},
        # A ragged batch of leaves (transpositions taken out) in half precision.
        {"name": "leaf_f16_b250", "kind": "leaf", "dtype": "f16", "batch": 250},
        # Many games played at once, one leaf each.
        {"name": "leaf_bf16_b1000", "kind": "leaf", "dtype": "bf16", "batch": 1000},
        # The e4m3 model serving a small ragged batch.
        {"name": "leaf_fp8_b33", "kind": "leaf", "dtype": "fp8", "batch": 33},
        # Self-play throughput, the headline configuration.
        {"name": "leaf_fp8_b4096", "kind": "leaf", "dtype": "fp8", "batch": 4096},
        # The GPT model asked for one move.
        {"name": "gpt_move_b1", "kind": "gpt_move", "dtype": "bf16", "batch": 1},
        # A file of positions labelled with the GPT model: FEN strings in, probabilities and moves on the host out.
        {"name": "gpt_fens_n1500", "kind": "gpt_fens", "dtype": "bf16", "batch": 1500},
        # Scoring half of a GRPO step: 8 x 16 sequences of 64 board and 192 move tokens, policy and reference model.
        {"name": "gpt_score_n128_t192", "kind": "gpt_score", "dtype": "bf16", "batch": 128, "tokens": 192},
        # Rollout half of a GRPO step: 8 x 16 sequences of 191 sampled tokens.
        {"name": "gpt_rollout_n128", "kind": "gpt_rollout", "dtype": "bf16", "batch": 128},
        # Validation pass of BT4 training: games of 31 positions with policy and value losses.
        {"name": "bt4_loss_16x31", "kind": "bt4_loss", "dtype": "bf16", "batch": 16, "seq": 31},
        # 1-ply value search over the games of an evaluation match: FEN strings in, move values on the host out.
        {"name": "bt4_search_n48", "kind": "bt4_search", "dtype": "bf16", "batch": 48},
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    kind = rng.choice(["leaf", "leaf", "leaf", "leaf", "gpt_move", "gpt_fens", "gpt_score", "gpt_rollout", "bt4_loss", "bt4_search"])
    if kind == "leaf":
        dtype = rng.choice(["bf16", "f16", "fp8"])
        return {"kind": kind, "dtype": dtype, "batch": size(1, 4096 if dtype == "fp8" else 2048)}
    if kind == "gpt_move":
        return {"kind": kind, "dtype": rng.choice(["bf16", "fp8"]), "batch": size(1, 2048)}
    if kind == "gpt_fens":
        return {"kind": kind, "dtype": rng.choice(["bf16", "fp8"]), "batch": size(1, 6000)}
    if kind == "gpt_score":
        return {"kind": kind, "dtype": "bf16", "batch": size(4, 128), "tokens": size(8, 192)}
    if kind == "gpt_rollout":
        return {"kind": kind, "dtype": "bf16", "batch": size(1, 128)}
    if kind == "bt4_loss":
        return {"kind": kind, "dtype": "bf16", "batch": size(1, 32), "seq": size(4, 64)}
    return {"kind": kind, "dtype": "bf16", "batch": size(1, 64)}


_MODELS = {}


def _model(name):
    """The process's one model of a kind; the e4m3 ones are calibrated on 512 positions."""
    if name not in _MODELS:
        kind, _, dtype = name.partition(":")
        kw = {"fp8": dtype == "fp8", "act_dtype": "f16" if dtype == "f16" else "bf16"}
        if kind == "leaf":
            m = models.BT4Class(LEAF_L, LEAF_C, LEAF_F, LEAF_H, seed=0, **kw)
        elif kind == "bt4":
            m = models.BT4(seed=0, **kw)
        else:
            cfg = models.GPTConfig(block_size=GPT_BLOCK, vocab_size=VOCAB_RL, n_layer=GPT_LAYERS, n_head=GPT_HEADS, n_embd=GPT_C)
            m = models.GPT(cfg, seed=1 if kind == "gpt_ref" else 0, **kw)
            if kind == "gpt_sure":
                m.load_state_dict(_sure(m.state_dict()))
        if kw["fp8"]:
            m.calibrate(torch.from_numpy(board.random_positions(2, 512)["planes"]).to(DEV))
        _MODELS[name] = m
    return _MODELS[name]


def _sure(sd):
    """Weights of a model that is sure of its next token, as a trained policy is: the positional rows behind the board
    carry the embedding of the token that follows, so nearly all mass lies on it (moves, now and then the end of a
    variation, </thinking> near the end). Rounding then moves single draws, it does not send whole sequences apart."""
    g = torch.Generator().manual_seed(5)
    steps = GPT_BLOCK - 65
    follow = torch.randint(0, START_THINK, (steps,), generator=g)
    follow[30:150:30] = END_VARIATION
    follow[170], follow[172:] = END_THINK, END
    sd["pe"][65:65 + steps] = 50.0 * sd["lm_head.weight"][follow]
    return sd


def prepare(case, seed):
    kind, n, dtype = case["kind"], case["batch"], case["dtype"]
    g = torch.Generator().manual_seed(seed)
    if kind == "leaf":
        r = board.random_positions(seed, n, late_fraction=0.3, masks_leela=True)
        return {"kind": kind, "model": _model("leaf:" + dtype), "planes": torch.from_numpy(r["planes"]).to(DEV),
                "mask": torch.from_numpy(r["masks_leela"]).to(DEV)}
    if kind == "gpt_move":
        planes = torch.from_numpy(board.random_positions(seed, n)["planes"]).to(DEV)
        return {"kind": kind, "model": _model("gpt:" + dtype), "planes": planes, "idx": torch.zeros((n, 0), dtype=torch.int64, device=DEV)}
    if kind == "gpt_fens":
        return {"kind": kind, "model": _model("gpt:" + dtype), "fens": board.random_positions(seed, n, planes=False, fens=True)["fens"]}
    if kind == "gpt_score":
        # eight sampled sequences per position, as a GRPO group
        planes = torch.from_numpy(board.random_positions(seed, -(-n // 8))["planes"]).to(DEV)
        planes = planes.repeat(8, 1, 1, 1)[:n].contiguous()
        seq = torch.randint(0, START_THINK, (n, case["tokens"]), generator=g).to(DEV)
        return {"kind": kind, "model": _model("gpt:" + dtype), "ref": _model("gpt_ref:" + dtype), "planes": planes, "seq": seq}
    if kind == "gpt_rollout":
        planes = torch.from_numpy(board.random_positions(seed, -(-n // 8))["planes"]).to(DEV)
        return {"kind": kind, "model": _model("gpt_sure:" + dtype), "planes": planes.repeat(8, 1, 1, 1)[:n].contiguous(), "seed": seed}
    if kind == "bt4_loss":
        s = case["seq"]
        planes = torch.from_numpy(board.random_positions(seed, n * s)["planes"]).to(DEV).reshape(n, s, 8, 8, 19)
        targets = torch.randint(0, START_THINK, (n, s), generator=g).to(DEV)
        values = torch.randint(0, 3, (n, s, 1), generator=g).to(DEV)
        return {"kind": kind, "model": _model("bt4:" + dtype), "inp": (planes, targets, None, values)}
    if kind == "bt4_search":
        return {"kind": kind, "model": _model("bt4:" + dtype), "fens": board.random_positions(seed, n, planes=False, fens=True)["fens"]}
    raise ValueError(kind)


def run(state):
    kind, m = state["kind"], state["model"]
    if kind == "leaf":
        return m.evaluate(state["planes"], legal_mask=state["mask"], T=1.0, want_probs=True)
    if kind == "gpt_move":
        return m.forward((state["planes"], state["idx"]))[0]
    if kind == "gpt_fens":
        probs, _, best = m.evaluate_fens(state["fens"])
        return probs, best
    if kind == "gpt_score":
        batch, seq = (state["planes"], state["seq"]), state["seq"]
        logits, loss, _ = m.forward(batch, compute_loss=True)
        ref = state["ref"].forward(batch, compute_loss=True)[0]
        mine, theirs = logits[:, 63:-1].reshape(-1, VOCAB_RL), ref[:, 63:-1].reshape(-1, VOCAB_RL)
        return (logits, loss) + models.token_scores(mine, seq.reshape(-1), theirs, want_kl=True)
    if kind == "gpt_rollout":
        return m.generate_sequence(state["planes"], T=1, seed=state["seed"])
    if kind == "bt4_loss":
        return m.forward(state["inp"], compute_loss=True)[:4]
    picks, per_root = m.get_best_moves_value(state["fens"], T=0.0, return_values=True)
    # (the picks as their values: equal values make equal picks)
    chosen = [float(v[mv.index(p)]) if p else 0.0 for p, (mv, v) in zip(picks, per_root)]
    values = torch.zeros(len(picks) * MOST_MOVES)
    flat = torch.cat([v for _, v in per_root])
    values[:flat.numel()] = flat
    return values, torch.tensor(chosen)


def _gpt_token():
    """2*MAC of one token through one GPT layer's linears."""
    return 24.0 * GPT_C * GPT_C


def work(case):
    kind, n, fp8 = case["kind"], case["batch"], case["dtype"] == "fp8"
    wb = 1 if fp8 else 2
    T = 64
    if kind == "leaf":
        C, F, L, H = LEAF_C, LEAF_F, LEAF_L, LEAF_H
        smol = 2 * T * C * 32 + 2 * 2048 * 256 + 2 * 256 * H * 256 + 2 * H * 256 * 4096
        heads = 6 * T * C * C + 2 * T * T * C + 2 * T * C * 128 + 2 * 8192 * 128 + 2 * T * 19 * C
        flops = L * (8 * T * C * C + 4 * T * T * C + 4 * T * C * F + smol) + heads
        weights = wb * (L * (4 * C * C + 2 * C * F + 32 * C) + 4096 * 256) + 2 * (L * (2048 * 256 + 256 * H * 256) + 3 * C * C + 128 * (C + 8192))
        return {"bytes": weights + n * (T * 19 * 4 + VOCAB_LEELA * 5 + 12), "flops": n * flops}
    if kind in ("gpt_move", "gpt_fens"):
        # the last layer's queries, projection and MLP are needed for one token only
        C, L = GPT_C, GPT_LAYERS
        flops = (L - 1) * (T * _gpt_token() + 2 * T * (T + 1) * C) + T * 4 * C * C + 20 * C * C + 4 * T * C + 2 * T * 19 * C + 2 * C * VOCAB_RL
        weights = wb * (12 * L * C * C + VOCAB_RL * C)
        io = T * 19 * 4 + VOCAB_RL * 4 if kind == "gpt_move" else 64 + VOCAB_RL * 4 + 4
        return {"bytes": weights + n * io, "flops": n * flops}
    if kind == "gpt_score":
        C, L = GPT_C, GPT_LAYERS
        T = 64 + case["tokens"]
        flops = L * (T * _gpt_token() + 2 * T * (T + 1) * C) + T * 2 * C * VOCAB_RL + 2 * 64 * 19 * C
        return {"bytes": 2 * wb * (12 * L * C * C + VOCAB_RL * C) + n * (64 * 19 * 4 + case["tokens"] * 20 + T * VOCAB_RL * 4), "flops": 2 * n * flops}
    if kind == "gpt_rollout":
        C, L, S = GPT_C, GPT_LAYERS, GPT_BLOCK - 65
        T = 64 + S
        flops = L * (T * _gpt_token() + 2 * T * (T + 1) * C) + S * 2 * C * VOCAB_RL + 2 * 64 * 19 * C
        return {"bytes": wb * (12 * L * C * C + VOCAB_RL * C) + n * (64 * 19 * 4 + (S + 1) * 8 + S * VOCAB_RL * 4), "flops": n * flops}
    C, F, L = BT4_C, BT4_F, BT4_L
    trunk = L * (8 * T * C * C + 6 * T * T * C + 4 * T * C * F) + 2 * T * 19 * C
    value = 2 * T * C * 128 + 2 * 8192 * 128
    weights = wb * L * (4 * C * C + 2 * C * F) + 2 * 128 * (C + 8192)
    if kind == "bt4_loss":
        n *= case["seq"]
        policy = 6 * T * C * C + 2 * T * T * C + 2 * 4096 * VOCAB_RL
        weights += 2 * (3 * C * C + 4096 * VOCAB_RL)
        return {"bytes": weights + n * (T * 19 * 4 + VOCAB_RL * 4 + 28), "flops": n * (trunk + value + policy)}
    return {"bytes": weights + n * (64 + CHILDREN * 4), "flops": n * CHILDREN * (trunk + value)}


def tolerance(case):
    """What two correct runs at the case's precision differ by. The post-LN encoders keep a 16-bit residual stream through
    all layers (bf16: 1.1e-2 on the value logits against an fp32 stream, BT4's policy 7e-3), GPT an fp32 one (logits
    2.5e-3); an e4m3 layer turns any other rounding into other codes (2.3e-2 between two ways to round the norms)."""
    kind, dtype = case["kind"], case["dtype"]
    if kind == "gpt_rollout":       # probabilities that lie nearly all on one token
        return {"rel": 1e-3, "max": 0.05, "differ": 3e-3}
    if dtype == "fp8":
        return {"rel": 3e-2, "max": 0.3, "differ": 1e-2}
    if kind == "bt4_search":        # values are probabilities near 1/2, the differences of logits average out
        return {"rel": 1e-3, "max": 5e-3}
    if kind.startswith("gpt"):
        return {"rel": 4e-3, "max": 0.05, "differ": 1e-2}
    return {"rel": 1.5e-2, "max": 0.15} if dtype == "bf16" else {"rel": 2e-3, "max": 0.02}
