"""The work whose speed is kept track of: calls of the VecMarket engine and of the
high-low game, through their public Python entry points, over the sizes in use.

Every case is one pass of a program that goes on: a market step, a replay of several
steps, a game step or a whole episode. A state keeps its books from pass to pass, as a
program's does, and is prepared past the point where the order ring has wrapped, so
that a pass inserts, matches and evicts as it does in the long run. Its quotes are a
block of steps that is played forwards and backwards in turn.

All outputs are whole numbers (or whole numbers as float32, and a few constants of the
observation), the results of an integer state machine: they are the same bit for bit, so
tolerance() is "exact", and there is no 64-bit reference that could be closer.
"""
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (ROOT, os.path.join(ROOT, "astra-cuda_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

BLOCK = 512  # steps of quotes a state keeps

# price levels, orders, fills and customers of a market
BOOK = {"levels": 128, "orders": 1024, "fills": 1024, "customers": 16}
DEEP = {"levels": 512, "orders": 4096, "fills": 4096, "customers": 64}
# the game's own market at its default parameters (5 players, 20 steps, prices to 30)
SMALL = {"levels": 31, "orders": 200, "fills": 10, "customers": 5}


def _quotes(name, markets, stream, book, layout="columns", binding="python"):
    return dict(name=name, kind="quotes", markets=markets, stream=stream, layout=layout, binding=binding, **book)


def listed():
    return [
        # The smallest: 64 markets of the CPU reference run. Nothing but latency and launches.
        _quotes("quotes_64", 64, "band", BOOK),
        # A thousand of the game's own small books, through the compiled binding.
        _quotes("quotes_1000_small_compiled", 1000, "uniform", SMALL, binding="compiled"),
        # The README's shape: 10,000 markets, half of the quotes cross, BBOs every step.
        _quotes("quotes_10k", 10_000, "uniform", BOOK),
        # The deep book: 512 levels, 4,096 orders, 64 customers.
        _quotes("deep_20k", 20_000, "normal", DEEP),
        # A ragged count in between, with the row layout of the fill batch.
        _quotes("quotes_33333_rows", 33_333, "walk", BOOK, layout="rows"),
        # The headline: 100,000 markets around a random walk, the drop-in calls.
        _quotes("quotes_100k", 100_000, "walk", BOOK),
        # The largest: 524,288 markets (25 GB of books and fills).
        _quotes("quotes_524k", 524_288, "walk", BOOK),
        # Replays: the quotes of many steps in hand, one launch, every step's counts and BBOs kept.
        dict(name="replay_10k", kind="replay", markets=10_000, steps=32, stream="uniform", layout="columns", **BOOK),
        dict(name="replay_100k_rows", kind="replay", markets=100_000, steps=16, stream="walk", layout="rows", **BOOK),
        # Markets that end and start anew: books cleared by a mask, quotes, BBOs, last prices
        # and the portfolios copied out, step by step.
        dict(name="auto_reset_30k", kind="auto_reset", markets=30_000, stream="walk", layout="columns", **BOOK),
        # One step of a policy in the high-low game at rollout size on a book of full size:
        # observation, checked move, rewards.
        dict(name="game_step_10k", kind="game_step", markets=10_000, players=5, steps=200, max_value=127,
             max_trade=5, max_size=5, levels=128, orders=1024, fills=10, customers=16, check=True),
        # The reference's game benchmark: an episode of 262,144 envs with its rollout kept.
        dict(name="game_episode_262k", kind="game_episode", markets=262_144, players=5, steps=8, max_value=10,
             max_trade=1, max_size=2, check=True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the ranges that the listed ones stand for."""
    kind = rng.choice(["quotes", "quotes", "quotes", "replay", "auto_reset", "game_step", "game_episode"])
    if kind in ("quotes", "replay", "auto_reset"):
        book, stream = dict(rng.choice([BOOK, BOOK, SMALL, DEEP])), rng.choice(["uniform", "walk", "band", "normal"])
        most = 20_000 if book["orders"] > 1024 else 200_000
        c = dict(kind=kind, markets=_log_int(rng, 40, most if kind != "replay" else most // 2), stream=stream,
                 layout=rng.choice(["columns", "columns", "rows"]), **book)
        if kind == "quotes":
            # (the compiled binding has the reference's fill batch and its limits on the shape)
            c["binding"] = rng.choice(["python", "compiled"]) if c["layout"] == "columns" and most > 20_000 else "python"
        if kind == "replay":
            c["steps"] = rng.randint(2, 32)
        return c
    players = rng.randint(4, 8)
    if kind == "game_step":
        return dict(kind=kind, markets=_log_int(rng, 100, 65_536), players=players, steps=rng.randint(20, 200),
                    max_value=rng.randint(10, 127), max_trade=rng.randint(1, 5), max_size=rng.randint(1, 5),
                    levels=128, orders=1024, fills=10, customers=16, check=rng.random() < 0.7)
    return dict(kind=kind, markets=_log_int(rng, 500, 65_536), players=players, steps=rng.randint(4, 10),
                max_value=rng.randint(5, 30), max_trade=rng.randint(1, 5), max_size=rng.randint(1, 5),
                check=rng.random() < 0.7)


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _ints(g, lo, hi, shape):
    """Whole numbers in [lo, hi]."""
    return torch.randint(lo, hi + 1, shape, generator=g, device="cuda", dtype=torch.int32)


def _stream(case, g):
    """BLOCK steps of quotes: five int32 [BLOCK, markets] tensors (bid price and size, ask price and size, customer)."""
    M, L, C = case["markets"], case["levels"], case["customers"]
    shape, kind = (BLOCK, M), case["stream"]
    cust = _ints(g, 0, C - 1, shape)
    bsz, asz = _ints(g, 1, 10, shape), _ints(g, 1, 10, shape)
    if kind == "band":  # a one-customer-at-a-time market; quotes rarely cross at once
        bid = _ints(g, 0, L // 2 - 1, shape)
        ask = torch.clamp(bid + _ints(g, 1, L // 2 - 1, shape), max=L - 1)
        cust = (torch.arange(BLOCK, device="cuda", dtype=torch.int32) % C).unsqueeze(1).repeat(1, M)
    elif kind == "uniform":  # half of the quotes cross
        bid, ask = _ints(g, 0, L - 1, shape), _ints(g, 0, L - 1, shape)
    elif kind == "walk":  # a random walk per market, a narrow spread, geometric sizes
        mid = torch.full((M,), L // 2, device="cuda", dtype=torch.int32)
        move = _ints(g, -3, 3, shape)
        mids = torch.empty(shape, device="cuda", dtype=torch.int32)
        for k in range(BLOCK):
            mid = torch.clamp(mid + move[k], 0, L - 1)
            mids[k] = mid
        spread = _ints(g, 0, 8, shape)
        bid = torch.clamp(mids - spread // 2, 0, L - 1)
        ask = torch.clamp(bid + spread, 0, L - 1)
        bsz = torch.empty(shape, device="cuda").geometric_(0.3, generator=g).clamp_(max=50).to(torch.int32)
        asz = torch.empty(shape, device="cuda").geometric_(0.3, generator=g).clamp_(max=50).to(torch.int32)
    else:  # "normal": prices around the middle of a deep book, larger sizes
        def price():
            x = torch.randn(shape, generator=g, device="cuda") * (L * 40.0 / 512.0) + L / 2.0
            return x.round_().clamp_(0, L - 1).to(torch.int32)
        bid, ask = price(), price()
        bsz, asz = _ints(g, 1, 100, shape), _ints(g, 1, 100, shape)
    return [t.contiguous() for t in (bid, bsz, ask, asz, cust)]


def _prepare_market(case, seed):
    if case.get("binding") == "compiled":
        from astra_cuda._C import order_matching as om
    else:
        from astra_cuda import order_matching as om
    g = _generator(seed)
    L, O, F, C = case["levels"], case["orders"], case["fills"], case["customers"]
    extended = {"allow_extended_shapes": True} if O > 1024 else {}
    market = om.VecMarket(case["markets"], L, O, F, C, 0, 64, **extended)
    fills = market.new_fill_batch(layout="rows") if case["layout"] == "rows" else market.new_fill_batch()
    bbos = market.new_bbo_batch()
    q = _stream(case, g)
    s = {"case": case, "market": market, "fills": fills, "bbos": bbos, "at": 0, "back": False}
    # past the ring's first wrap: two orders a step
    for i in range(O // 2 // BLOCK + 1):
        turned = q if i % 2 == 0 else [torch.flip(t, (0,)) for t in q]
        for k in range(BLOCK):
            market.add_two_sided_quotes(*(t[k] for t in turned), fills)
    s["back"] = O // 2 // BLOCK % 2 == 0
    s["at"] = BLOCK - 1 if s["back"] else 0
    if case["kind"] == "replay":
        n, M = case["steps"], case["markets"]
        blocks = [[t[i:i + n].contiguous() for t in q] for i in range(0, BLOCK - n + 1, n)]
        s["blocks"], s["at"], s["back"] = blocks, len(blocks) - 1, True
        s["counts"] = torch.zeros((n, M), dtype=torch.int32, device="cuda")
        s["step_bbos"] = torch.zeros((4, n, M), dtype=torch.int32, device="cuda")
    else:
        s["steps"] = [tuple(t[k] for t in q) for k in range(BLOCK)]
    if case["kind"] == "auto_reset":
        s["ended"] = list((torch.rand((BLOCK, case["markets"]), generator=g, device="cuda") < 1 / 64).unbind(0))
        s["portfolios"] = torch.zeros((case["markets"], C, 2), dtype=torch.int32, device="cuda")
    return s


def _next(s, items):
    """The next of `items`, forwards and backwards in turn."""
    i = s["at"]
    if s["back"]:
        s["at"], s["back"] = (i - 1, True) if i > 0 else (0, False)
    else:
        s["at"], s["back"] = (i + 1, False) if i + 1 < len(items) else (i, True)
    return items[i], i


def _fields(fills):
    return [fills.fill_prices, fills.fill_sizes, fills.fill_customer_ids, fills.fill_quoter_ids,
            fills.fill_is_sell_quote, fills.fill_quote_sizes, fills.fill_tid, fills.fill_quote_tid, fills.fill_counts]


def _bbo_fields(b):
    return [b.best_bid_prices, b.best_bid_sizes, b.best_ask_prices, b.best_ask_sizes]


def _prepare_game(case, seed):
    import astra_cuda as astra
    g = _generator(seed)
    N, P, T, V = case["markets"], case["players"], case["steps"], case["max_value"]
    astra.register_games()
    params = {"steps_per_player": T, "max_contracts_per_trade": case["max_trade"],
              "customer_max_size": case["max_size"], "max_contract_value": V, "players": P, "num_markets": N,
              "threads_per_block": 256, "device_id": 0, "check_moves": case["check"]}
    if "levels" in case:
        params.update(market_price_levels=case["levels"], market_orders=case["orders"],
                      market_fills=case["fills"], market_customers=case["customers"])
    game = astra.load_game("high_low_trading", params)
    state = game.new_initial_state()
    signs = _ints(g, 0, 1, (N, P - 3)) * 2 - 1
    chance = [_ints(g, 1, V, (N, 2)), _ints(g, 0, 1, (N,)),
              torch.rand((N, P), generator=g, device="cuda").argsort(1).to(torch.int32),
              signs * _ints(g, 1, case["max_size"], (N, P - 3))]
    moves = min(P * T, 256)
    actions = torch.empty((moves, N, 4), dtype=torch.int32, device="cuda")
    actions[:, :, 0:2] = _ints(g, 1, V, (moves, N, 2))
    actions[:, :, 2:4] = _ints(g, 0, case["max_trade"], (moves, N, 2))
    s = {"case": case, "game": game, "state": state, "chance": chance, "actions": list(actions.unbind(0)), "at": 0}
    n = P * T if case["kind"] == "game_episode" else 1
    s["obs"] = torch.zeros([n] + game.observation_tensor_shape(), dtype=torch.float32, device="cuda")
    s["rewards"] = torch.zeros((n, N, P), dtype=torch.float32, device="cuda")
    s["since"] = torch.zeros((n, N), dtype=torch.float32, device="cuda")
    s["returns"] = torch.zeros((N, P), dtype=torch.float32, device="cuda")
    if case["kind"] == "game_step":  # into the middle of an episode
        _deal(s)
        for _ in range(P * T * 3 // 5):
            state.apply_action(s["actions"][s["at"] % moves])
            s["at"] += 1
    return s


def _deal(s):
    s["state"].reset()
    for a in s["chance"]:
        s["state"].apply_action(a)
    s["at"] = 0


def _game_step(s, row):
    state, obs, rewards, since = s["state"], s["obs"][row], s["rewards"][row], s["since"][row]
    player = state.current_player()
    state.fill_observation_tensor(obs)
    state.apply_action(s["actions"][s["at"] % len(s["actions"])])
    state.fill_rewards(rewards)
    state.fill_rewards_since_last_action(since, player)
    s["at"] += 1


def prepare(case, seed):
    return _prepare_game(case, seed) if case["kind"].startswith("game") else _prepare_market(case, seed)


def run(s):
    kind = s["case"]["kind"]
    if kind == "game_step":
        if s["state"].is_terminal():
            _deal(s)
        _game_step(s, 0)
        return [s["obs"], s["rewards"], s["since"], s["state"].market.get_customer_portfolios(),
                s["state"].bbo_batch.last_prices] + _bbo_fields(s["state"].bbo_batch)
    if kind == "game_episode":
        _deal(s)
        k = 0
        while not s["state"].is_terminal():
            _game_step(s, k)
            k += 1
        s["state"].fill_returns(s["returns"])
        return [s["obs"], s["rewards"], s["since"], s["returns"], s["state"].market.get_customer_portfolios(),
                s["state"].bbo_batch.last_prices] + _bbo_fields(s["state"].bbo_batch)
    market, fills, bbos = s["market"], s["fills"], s["bbos"]
    if kind == "replay":
        q, _ = _next(s, s["blocks"])
        market.add_two_sided_quotes_steps(*q, fills, s["counts"], s["step_bbos"])
        return _fields(fills) + [s["counts"], s["step_bbos"], market.get_customer_portfolios()]
    q, i = _next(s, s["steps"])
    if kind == "auto_reset":
        market.clear_quotes(s["ended"][i])
    market.add_two_sided_quotes(*q, fills)
    market.get_bbos(bbos)
    out = _fields(fills) + _bbo_fields(bbos)
    if kind == "auto_reset":
        bbos.update_last_prices(fills)
        market.copy_customer_portfolios_to(s["portfolios"])
        return out + [bbos.last_prices, s["portfolios"]]
    return out + [market.get_customer_portfolios()]


# Fills and emptied levels of a market in a step, about, per kind of stream.
FILLS = {"band": 0.9, "uniform": 1.3, "walk": 1.5, "normal": 1.4}
EMPTIED = {"band": 0.9, "uniform": 1.3, "walk": 0.95, "normal": 1.3}


def work(case):
    """Per market and step: 20 bytes of quotes and 4 of the count, 32 per inserted order (its record, its
    level's tail, a link), 109 per fill (29 of the row, two heads' records, two sizes, two portfolios, two
    links), 8 per emptied level, 24 for the BBO. No floating operations."""
    M = case["markets"]
    if case["kind"].startswith("game"):
        P = case["players"]
        fills = min(0.5 * case["max_trade"], 1.0)
        # the move and its market, the portfolios before and after, telemetry and rewards; the observation
        # written and its columns read; both rewards read and written as float32
        step = 16 + 16 * P + 56 + 24 * P + 24 + 32 * 1.6 + (109 + 8) * fills
        step += 4 * (12 + 6 * P) + 24 * P + 25 + 8 * P + 8
        n = P * case["steps"] if case["kind"] == "game_episode" else 1
        return {"bytes": M * step * n, "flops": 0}
    step = 24 + 24 + 32 * 2 + 109 * FILLS[case["stream"]] + 8 * EMPTIED[case["stream"]]
    if case["kind"] == "auto_reset":
        # the mask; a cleared market's levels; the last prices; the portfolios read and written
        step += 1 + 8 * case["levels"] / 64 + 8 + 16 * case["customers"]
    return {"bytes": M * step * case.get("steps", 1), "flops": 0}


def tolerance(case):
    return "exact"
