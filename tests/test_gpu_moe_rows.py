"""The experts' products on the matrix cores, each form over the same rows: few rows an expert (tiles of up to 64, the matrix
straight from memory), whole tiles of the walk that brings both operands straight into LDS (up to 64, 128 and 256 rows), whole tiles
staged through registers (up to 128, rows that begin at any offset).  Every class of rows a tile, K of one step and of many, columns that do not fill a fragment."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("k, n_out", [(32, 16), (96, 40), (512, 65), (1056, 130), (2432, 2560)])
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("more", [1, 4])
def test_every_form_against_float64(k, n_out, gated, more):
    import torch
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(k + n_out)
    counts = [1, 0, 16, 17, 33, 64, 65, 130, 5] if more == 1 else [300, 97, 128, 0, 257, 31, 192, 220]
    experts, rows = len(counts), sum(counts)
    order = rng.permutation(rows).astype(np.int32)
    x = torch.tensor(rng.normal(size=(rows, k)).astype(np.float32), device=DEV).bfloat16()
    w = torch.tensor((rng.normal(size=(experts, n_out * (2 if gated else 1), k)) * k ** -0.5).astype(np.float32), device=DEV).bfloat16()
    weight = torch.tensor(rng.uniform(0.2, 1.0, size=rows).astype(np.float32), device=DEV)
    gather = torch.tensor(order, device=DEV)
    starts = np.concatenate([[0], np.cumsum(counts)[:-1]])
    # float64 of what the bfloat16 operands hold
    xd, wd = x.double()[gather.long()], w.double()
    ref = torch.empty((rows, n_out), dtype=torch.float64, device=DEV)
    size = torch.empty_like(ref)
    for e, (at, n) in enumerate(zip(starts, counts)):
        p = xd[at:at + n] @ wd[e].T
        a = xd[at:at + n].abs() @ wd[e].abs().T
        if gated:
            s = weight[at:at + n].double()[:, None]
            g, u = s * p[:, :n_out], s * p[:, n_out:]
            ref[at:at + n] = g * torch.sigmoid(g) * u
            size[at:at + n] = 1.1 * s * a[:, :n_out] * u.abs() + (g * torch.sigmoid(g)).abs() * s * a[:, n_out:]     # |silu'| < 1.1
        else:
            ref[at:at + n], size[at:at + n] = torch.relu(p), a
    for tile_rows, offset in ((64, 0), (128, 0), (256, 0), (128, 1)):
        tiles = [(e, at + j, min(tile_rows, n - j)) for e, (at, n) in enumerate(zip(starts, counts)) for j in range(0, n, tile_rows)] + [(0, 0, 0)] * 3
        td = torch.tensor(np.array(tiles, dtype=np.int32), device=DEV)
        for through in (gather, None):
            xs = x if through is not None else x[gather.long()].contiguous()
            if offset:          # rows that begin at no multiple of 16 bytes: the staged kernel
                flat = torch.empty(rows * k + 8, dtype=torch.bfloat16, device=DEV)
                xs = flat[offset:offset + rows * k].view(rows, k).copy_(xs)
            for ty in (torch.float32, torch.bfloat16):
                out = torch.full((rows, n_out), float("nan"), dtype=ty, device=DEV)
                if gated:
                    ops.moe_expert_gated(xs, through, weight, w, td, out, "silu", tile_rows=tile_rows)
                else:
                    ops.moe_expert(xs, through, w, td, out, "relu", tile_rows=tile_rows)
                # sums of k exact products in float32, in any order, and one rounding of the result
                bound = (k + 4) * 2.0 ** -24 * size + (2.0 ** -8 if ty == torch.bfloat16 else 2.0 ** -22) * ref.abs() + 1e-30
                assert bool(((out.double() - ref).abs() <= bound).all()), (tile_rows, offset, ty)


@pytest.mark.parametrize("tile_rows", [64, 128, 256])
def test_the_sort_shares_rows_out(tile_rows):
    """Every sorted row in one tile of its expert, tiles no larger than asked for, used ones first."""
    import torch
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(tile_rows)
    tokens, experts, top = 1500, 7, 2
    z = rng.normal(size=(tokens, experts)).astype(np.float32)
    z[:, 0] += 1.5
    z[:, 3] = -30.0
    new = lambda *shape: torch.empty(shape, dtype=torch.int32, device=DEV)  # noqa: E731
    chosen, weight, pair_token, place = new(tokens, top), torch.empty((tokens, top), device=DEV), new(tokens * top), new(tokens * top)
    tiles = new(ops.moe_max_tiles(tokens, experts, top, tile_rows), 3)
    ops.moe_route(torch.tensor(z, device=DEV), experts, top, 1e-20, chosen, weight, pair_token, place, tiles, tile_rows=tile_rows)
    expert_of_row = np.empty(tokens * top, dtype=int)
    expert_of_row[place.cpu().numpy().reshape(-1)] = chosen.cpu().numpy().reshape(-1)
    covered = np.zeros(tokens * top, dtype=int)
    listed = tiles.cpu().numpy()
    assert np.all(np.diff((listed[:, 2] > 0).astype(int)) <= 0)
    for e, first, n in listed:
        assert 0 <= n <= tile_rows and np.all(expert_of_row[first:first + n] == e)
        covered[first:first + n] += 1
    assert np.all(covered == 1)


@pytest.mark.parametrize("experts, tokens", [(5, 1), (64, 4), (64, 5), (65, 4), (200, 16), (200, 17), (257, 3)])
def test_choice_and_sort_in_one_launch_and_in_two(experts, tokens):
    """On both sides of the tokens and experts up to which one launch chooses and sorts: the choices of the written-out softmax, every
    pair in a row of its expert's run, the runs in the order of the experts."""
    import torch
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(experts + tokens)
    top = 4
    z = rng.normal(size=(tokens, experts)).astype(np.float32)
    new = lambda *shape: torch.full(shape, -7, dtype=torch.int32, device=DEV)  # noqa: E731
    for grouped in (False, True):
        chosen, weight, pair_token, place = new(tokens, top), torch.empty((tokens, top), device=DEV), new(tokens * top), new(tokens * top)
        tiles = new(ops.moe_max_tiles(tokens, experts, top, 64), 3)
        ops.moe_route(torch.tensor(z, device=DEV), experts, top, 1e-20, chosen, weight, pair_token, place, tiles, tile_rows=64,
                      router="sigmoid" if grouped else "softmax")
        picked = np.argsort(-z, axis=1, kind="stable")[:, :top]
        assert np.array_equal(chosen.cpu().numpy(), picked)
        s = np.take_along_axis(1 / (1 + np.exp(-z.astype(np.float64))) if grouped else np.exp(z.astype(np.float64)), picked, axis=1)
        assert np.allclose(weight.cpu().numpy(), s / s.sum(axis=1, keepdims=True), rtol=1e-5)      # float32 exponentials, a few of them
        at = place.cpu().numpy()
        assert np.array_equal(np.sort(at), np.arange(tokens * top))
        assert np.array_equal(pair_token.cpu().numpy()[at], np.arange(tokens * top) // top)
        expert_of_row = np.empty(tokens * top, dtype=int)
        expert_of_row[at] = picked.reshape(-1)
        assert np.all(np.diff(expert_of_row) >= 0)
        listed = tiles.cpu().numpy()
        used = listed[listed[:, 2] > 0]
        assert np.array_equal(np.repeat(used[:, 0], used[:, 2]), expert_of_row) and np.array_equal(np.cumsum(used[:, 2]) - used[:, 2], used[:, 1])


def test_operands_at_any_offset():
    """Rows that begin at no multiple of 16 bytes take the staged kernel, whatever the rows an expert: as if they lay at one."""
    import torch
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(2)
    rows, k, n_out = 120, 96, 64
    flat = torch.tensor(rng.normal(size=rows * k + 8), dtype=torch.bfloat16, device=DEV)
    w = torch.tensor(rng.normal(size=(1, n_out, k)), dtype=torch.bfloat16, device=DEV)
    tiles = torch.tensor([[0, 0, rows]], dtype=torch.int32, device=DEV)
    results = []
    for x in (flat[2:2 + rows * k].view(rows, k), flat[2:2 + rows * k].view(rows, k).clone()):
        results.append(ops.moe_expert(x, None, w, tiles, torch.empty((rows, n_out), device=DEV), tile_rows=128))
    ref = flat[2:2 + rows * k].view(rows, k).double() @ w[0].double().T
    size = flat[2:2 + rows * k].view(rows, k).double().abs() @ w[0].double().abs().T
    for out in results:
        assert bool(((out.double() - ref).abs() <= (k + 4) * 2.0 ** -24 * size).all())


@pytest.mark.parametrize("k, n_out", [(512, 1040), (1024, 528), (1056, 528)])
@pytest.mark.parametrize("gated", [False, True])
def test_lists_of_few_rows_in_products_of_little_k(k, n_out, gated):
    """On both sides of the K up to which a launch of many workgroups takes the walk for tiles of up to 64 rows: lists of 64
    and of 128 rows against float64."""
    import torch
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(k)
    counts = list(rng.integers(0, 9, 64)) + [64, 33, 65, 17]
    experts, rows = len(counts), int(sum(counts))
    x = torch.tensor(rng.normal(size=(rows, k)).astype(np.float32), device=DEV).bfloat16()
    w = torch.tensor((rng.normal(size=(experts, n_out * (2 if gated else 1), k)) * k ** -0.5).astype(np.float32), device=DEV).bfloat16()
    starts = np.concatenate([[0], np.cumsum(counts)[:-1]])
    ref = torch.empty((rows, n_out), dtype=torch.float64, device=DEV)
    size = torch.empty_like(ref)
    for e, (at, n) in enumerate(zip(starts, counts)):
        p, a = x[at:at + n].double() @ w[e].double().T, x[at:at + n].double().abs() @ w[e].double().abs().T
        if gated:
            g, u = p[:, :n_out], p[:, n_out:]
            ref[at:at + n] = torch.relu(g) * u
            size[at:at + n] = a[:, :n_out] * u.abs() + g.abs() * a[:, n_out:]
        else:
            ref[at:at + n], size[at:at + n] = p, a
    for tile_rows in (64, 128):
        tiles = [(e, at + j, min(tile_rows, n - j)) for e, (at, n) in enumerate(zip(starts, counts)) for j in range(0, n, tile_rows)] + [(0, 0, 0)] * 3
        td = torch.tensor(np.array(tiles, dtype=np.int32), device=DEV)
        out = torch.full((rows, n_out), float("nan"), device=DEV)
        if gated:
            ops.moe_expert_gated(x, None, None, w, td, out, "relu", tile_rows=tile_rows)
        else:
            ops.moe_expert(x, None, w, td, out, tile_rows=tile_rows)
        # sums of k exact products in float32, in any order
        assert bool(((out.double() - ref).abs() <= (k + 4) * 2.0 ** -24 * size + 2.0 ** -22 * ref.abs()).all()), tile_rows


def both_products(experts, width, inner, top, tokens, gated, tile_rows):
    """Milliseconds of 12 runs of a step's two products with tiles of so many rows, the best of six times."""
    import torch
    from kipp_amd.csrc import ops
    torch.manual_seed(tokens)
    pairs = tokens * top
    i32 = lambda *shape: torch.empty(shape, dtype=torch.int32, device=DEV)  # noqa: E731
    bf = lambda *shape: torch.randn(*shape, device=DEV).bfloat16()  # noqa: E731
    x, up, down = bf(tokens, width), bf(experts, inner * (2 if gated else 1), width), bf(experts, width, inner)
    mid, out = bf(pairs, inner), torch.empty((pairs, width), device=DEV)
    pair_token, place, tiles = i32(pairs), i32(pairs), i32(ops.moe_max_tiles(tokens, experts, top, tile_rows), 3)
    z = torch.randn(tokens, experts, device=DEV) + 0.4 * torch.randn(experts, device=DEV)
    ops.moe_route(z, experts, top, 1e-20, i32(tokens, top), torch.empty((tokens, top), device=DEV), pair_token, place, tiles, tile_rows=tile_rows)
    marks = []
    for _ in range(7):
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        begin.record()
        for _ in range(12):
            if gated:
                ops.moe_expert_gated(x, pair_token, None, up, tiles, mid, "silu", tile_rows=tile_rows)
            else:
                ops.moe_expert(x, pair_token, up, tiles, mid, "gelu", tile_rows=tile_rows)
            ops.moe_expert(mid, None, down, tiles, out, tile_rows=tile_rows)
        end.record()
        marks.append((begin, end))
    torch.cuda.synchronize()
    return min(a.elapsed_time(b) for a, b in marks[1:])


@pytest.mark.parametrize("experts, width, inner, top, tokens, gated, rows", [
    (256, 1024, 512, 8, 333, True, 256), (64, 2048, 704, 6, 128, False, 128), (32, 4096, 3072, 4, 96, True, 256), (8, 1024, 1024, 2, 1128, False, 128),
    (1, 4096, 3072, 1, 6, False, 64), (3, 4096, 768, 2, 13, False, 64), (16, 2048, 2432, 4, 33, True, 64), (32, 2560, 2432, 4, 96, False, 256),
    (32, 2560, 2432, 4, 1000, True, 256), (256, 512, 704, 4, 187, True, 64)])
def test_the_tiles_chosen_are_not_much_slower_than_others(experts, width, inner, top, tokens, gated, rows):
    """A step's choice beside the other tiles that its products could take, away from 32 experts of 2,432 x 2,560 and there."""
    import torch
    from kipp_amd.csrc import ops
    assert rows == ops.moe_tile_rows(torch.bfloat16, width, inner, pairs=tokens * top, experts=experts, gated=gated)
    took = {r: both_products(experts, width, inner, top, tokens, gated, r) for r in (64, 128, 256)}
    assert took[rows] <= 1.12 * min(took.values()), (rows, took)


@pytest.mark.parametrize("tokens", [1, 40, 700])
@pytest.mark.parametrize("gated", [False, True])
def test_feed_forward_of_rows_at_any_offset(tokens, gated):
    """The whole part over rows that begin at no multiple of 16 bytes: for steps of few pairs an expert, of some and of many."""
    import torch
    from kipp_amd.config import RoutedMLPSpec
    from kipp_amd.parts import build_part
    from kipp_amd.runtime import Runtime
    rng = np.random.default_rng(tokens)
    width, inner = 96, 16512 if gated else 33024        # (columns enough for tiles of 256 rows at so few experts)
    spec = RoutedMLPSpec(hidden_size=width, experts=3, top=2, expert_size=inner, activation="silu" if gated else "relu2", gate_name="gate" if gated else None)
    part = build_part("feed_forward", spec, Runtime("bfloat16"))
    part.load({name: torch.tensor(rng.normal(size=p.shape) / np.sqrt(p.shape[-1]), dtype=torch.bfloat16, device=DEV) for name, p in part.params(spec).items()})
    flat = torch.tensor(rng.normal(size=tokens * width + 8), dtype=torch.bfloat16, device=DEV)
    x = flat[1:1 + tokens * width].view(tokens, width)
    got, ref = part.forward(x), part.forward(x.clone())
    # the products in two orders of their sums, the inner rows rounded to bfloat16 in between
    assert float((got - ref).norm() / ref.norm()) < 4e-3


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("k, n_out", [(32, 2040), (96, 1160), (160, 900)])
def test_the_walk_over_many_tiles(gated, k, n_out):
    """Experts of one to three tiles in every number of fragments, and of none, with more workgroups than compute units: whole rounds, and what is left
    in halves of the columns (or not).  Small whole numbers, so that the sums are exact in any order."""
    import torch
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(k + n_out)
    sizes = [0, 1, 63, 64, 65, 128, 129, 192, 193, 256, 257, 300, 520]
    counts = [int(rng.choice(sizes)) for _ in range(33)]
    starts = np.cumsum([0] + counts[:-1])
    rows = int(np.sum(counts))
    x = torch.tensor(rng.integers(-3, 4, size=(rows, k)), dtype=torch.bfloat16, device=DEV)
    w = torch.tensor(rng.integers(-2, 3, size=(33, (2 if gated else 1) * n_out, k)), dtype=torch.bfloat16, device=DEV)
    weight = torch.tensor(rng.integers(1, 3, size=rows), dtype=torch.float32, device=DEV)
    tiles = []
    for e, (at, n) in enumerate(zip(starts, counts)):
        parts = -(-n // 256)
        each = -(-(-(-n // parts)) // 64) * 64 if parts else 0
        tiles += [(e, at + j * each, min(each, n - j * each)) for j in range(parts)]
    td = torch.tensor(np.array(tiles + [(0, 0, 0)] * 70, dtype=np.int32), device=DEV)
    out = torch.full((rows, n_out), float("nan"), device=DEV)
    if gated:
        ops.moe_expert_gated(x, None, weight, w, td, out, "relu", tile_rows=256)
    else:
        ops.moe_expert(x, None, w, td, out, tile_rows=256)
    for e, (at, n) in enumerate(zip(starts, counts)):
        p = x[at:at + n].float() @ w[e].float().T
        if gated:
            s = weight[at:at + n, None]
            p = torch.relu(s * p[:, :n_out]) * (s * p[:, n_out:])
        assert torch.equal(out[at:at + n], p), (e, n)


@pytest.mark.parametrize("order", ["mixed", "largest first", "gaps", "two in turn"])
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("tile_rows", [64, 128, 256])
def test_lists_of_tiles_in_any_order(order, gated, tile_rows):
    """Tiles of one expert that do not lie side by side in the list, and unused ones between them: every tile is done once, with its own expert's
    matrix.  Small whole numbers, so that the sums are exact in any order."""
    import torch
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(tile_rows)
    k, n_out, experts = 96, 1160, 33
    counts = [int(rng.choice([0, 1, 64, 65, 130, 257, 520])) for _ in range(experts)]
    starts = np.cumsum([0] + counts[:-1])
    rows = int(np.sum(counts))
    x = torch.tensor(rng.integers(-3, 4, size=(rows, k)), dtype=torch.bfloat16, device=DEV)
    w = torch.tensor(rng.integers(-2, 3, size=(experts, (2 if gated else 1) * n_out, k)), dtype=torch.bfloat16, device=DEV)
    tiles = [(e, at + j, min(tile_rows, n - j)) for e, (at, n) in enumerate(zip(starts, counts)) for j in range(0, n, tile_rows)]
    if order == "largest first":
        tiles.sort(key=lambda t: -t[2])
    elif order == "two in turn":
        tiles = tiles[0::2] + tiles[1::2]
    else:
        tiles = [tiles[i] for i in rng.permutation(len(tiles))]
    if order == "gaps":
        tiles = [t for tile in tiles for t in ((0, 0, 0), tile)] + [(0, 0, 0)] * 70
    td = torch.tensor(np.array(tiles, dtype=np.int32), device=DEV)
    out = torch.full((rows, n_out), float("nan"), device=DEV)
    if gated:
        ops.moe_expert_gated(x, None, None, w, td, out, "relu", tile_rows=tile_rows)
    else:
        ops.moe_expert(x, None, w, td, out, tile_rows=tile_rows)
    for e, (at, n) in enumerate(zip(starts, counts)):
        p = x[at:at + n].float() @ w[e].float().T
        if gated:
            p = torch.relu(p[:, :n_out]) * p[:, n_out:]
        assert torch.equal(out[at:at + n], p), (e, n)


@pytest.mark.parametrize("k, n_out, each, gated", [(384, 704, 2, True), (256, 2048, 12, False)])
def test_many_tiles_of_few_rows_share_compute_units(k, n_out, each, gated):
    """Products of little K over many tiles of up to 64 rows are their starts and ends, which two workgroups a compute unit hide from each other: faster than
    the same tiles where larger ones may come (level with those, and slower than the staged kernel, where they had a compute unit each)."""
    import torch
    from kipp_amd.csrc import ops
    experts = 256
    x = torch.randn(experts * each, k, device=DEV).bfloat16()
    w = torch.randn(experts, (2 if gated else 1) * n_out, k, device=DEV).bfloat16()
    td = torch.tensor([(e, e * each, each) for e in range(experts)], dtype=torch.int32, device=DEV)
    out = torch.empty(experts * each, n_out, dtype=torch.bfloat16, device=DEV)

    def run(rows):
        if gated:
            ops.moe_expert_gated(x, None, None, w, td, out, "silu", tile_rows=rows)
        else:
            ops.moe_expert(x, None, w, td, out, "silu", tile_rows=rows)
        return out
    assert torch.equal(run(64).clone(), run(128))
    took = {64: [], 128: []}
    for _ in range(6):
        for rows in took:
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            for _ in range(20):
                run(rows)
            end.record()
            took[rows].append((begin, end))
    torch.cuda.synchronize()
    few, whole = (min(a.elapsed_time(b) for a, b in took[rows]) for rows in (64, 128))
    assert few < 0.9 * whole, (few, whole)


@pytest.mark.parametrize("inner", [8, 7])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", ["silu", "gelu", "gelu_tanh"])
def test_activations_over_their_range(name, dtype, inner):
    """Where exponentials vanish, overflow and cancel, infinities and NaN, four columns a thread and one: within the rounding of the result and of
    float32 arithmetic (1 + erf and its like cancel below zero: an absolute error of some 2^-24 times z)."""
    import torch
    from kipp_amd.csrc import ops
    x = torch.cat([torch.linspace(-20, 20, 4001), torch.logspace(-30, 38, 700), -torch.logspace(-30, 38, 700), torch.randn(2207)]).float()
    x = x[:x.numel() // 56 * 56].reshape(-1, inner)
    got = ops.activate(x.to(DEV), torch.empty(x.shape, dtype=getattr(torch, dtype), device=DEV), name).cpu().double()
    z = x.double()
    u = 0.79788456080286535588 * (z + 0.044715 * z * z * z)
    ref = z * {"silu": torch.sigmoid(z), "gelu": torch.special.ndtr(z), "gelu_tanh": torch.sigmoid(2 * u)}[name]
    bound = 2.0 ** -22 * ref.abs() + 2.0 ** -23 * z.abs().clamp(max=20) + (2.0 ** -8 * ref.abs() if dtype == "bfloat16" else 0) + 1e-37
    assert bool(((got - ref).abs() <= bound).all())
    ends = torch.tensor([[float("inf"), float("nan"), 0.0, -3e38] + [1.0] * (inner - 4)])
    out = ops.activate(ends.to(DEV), torch.empty(ends.shape, dtype=getattr(torch, dtype), device=DEV), name).cpu()[0]
    assert out[0] == float("inf") and torch.isnan(out[1]) and out[2] == 0 and out[3] == 0


@pytest.mark.parametrize("router", ["softmax", "sigmoid"])
@pytest.mark.parametrize("tokens, experts, top, parts", [(16, 32, 32, 1), (4, 64, 32, 5), (1, 1, 1, 6), (16, 24, 1, 2), (5, 25, 1, 1), (16, 48, 2, 3), (17, 49, 2, 4),
                                                          (1024, 40, 4, 2), (1025, 40, 4, 1), (2048, 40, 4, 1), (2049, 64, 4, 2), (4096, 33, 4, 1), (4097, 33, 4, 3)])
def test_choices_and_places_at_the_edges_of_the_sort(router, tokens, experts, top, parts):
    """Numbers of pairs on both sides of what a thread of the sort keeps, of experts on both sides of choices by rank, as many choices as experts,
    equal scores, one to six slabs."""
    import torch
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(tokens + experts)
    z = rng.integers(-8, 9, size=(parts, tokens, experts)).astype(np.float32) / 8      # sums without rounding, many of them equal
    new = lambda *shape: torch.full(shape, -7, dtype=torch.int32, device=DEV)  # noqa: E731
    chosen, weight, pair_token, place = new(tokens, top), torch.empty((tokens, top), device=DEV), new(tokens * top), new(tokens * top)
    tiles = new(ops.moe_max_tiles(tokens, experts, top, 64), 3)
    ops.moe_route(torch.tensor(z if parts > 1 else z[0], device=DEV), experts, top, 1e-20, chosen, weight, pair_token, place, tiles, tile_rows=64, router=router)
    total = z.sum(0).astype(np.float64)
    picked = np.argsort(-total, axis=1, kind="stable")[:, :top]
    assert np.array_equal(chosen.cpu().numpy(), picked)
    s = np.take_along_axis(np.exp(total) if router == "softmax" else 1 / (1 + np.exp(-total)), picked, axis=1)
    assert np.allclose(weight.cpu().numpy(), s / s.sum(axis=1, keepdims=True), rtol=1e-5)      # float32 exponentials, up to 64 of them
    at = place.cpu().numpy()
    assert np.array_equal(np.sort(at), np.arange(tokens * top))
    assert np.array_equal(pair_token.cpu().numpy()[at], np.arange(tokens * top) // top)
    expert_of_row = np.empty(tokens * top, dtype=int)
    expert_of_row[at] = picked.reshape(-1)
    assert np.all(np.diff(expert_of_row) >= 0)


@pytest.mark.parametrize("k, n_out", [(1024, 530), (1056, 530), (1088, 513), (1504, 515), (1984, 520), (2048, 516), (2112, 528), (2432, 560), (2560, 512), (2624, 514), (4128, 516)])
@pytest.mark.parametrize("gathered", [False, True])
def test_few_tokens_have_the_bits_of_more(k, n_out, gathered):
    """A caller that says how few rows a tile has gets the numbers of one that does not, also where it is wrong: both sides of the K whose tiles have a
    kernel of their own, ends of the columns, rows at the edges of 16."""
    import torch
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(k)
    counts = [1, 2, 15, 16, 17, 0, 33, 64] + [1] * 40
    experts, rows = len(counts), int(sum(counts))
    starts = np.concatenate([[0], np.cumsum(counts)[:-1]])
    tiles = torch.tensor([(e, int(at), n) for e, (at, n) in enumerate(zip(starts, counts))] + [(0, 0, 0)] * 3, dtype=torch.int32, device=DEV)
    w = torch.tensor((rng.normal(size=(experts, n_out, k)) * k ** -0.5).astype(np.float32), device=DEV).bfloat16()
    x = torch.tensor(rng.normal(size=(29 if gathered else rows, k)).astype(np.float32), device=DEV).bfloat16()
    gather = torch.tensor(rng.integers(0, 29, rows), dtype=torch.int32, device=DEV) if gathered else None
    for dtype, act in ((torch.bfloat16, "relu2"), (torch.float32, None)):
        want = ops.moe_expert(x, gather, w, tiles, torch.empty((rows, n_out), dtype=dtype, device=DEV), act, tile_rows=64)
        got = ops.moe_expert(x, gather, w, tiles, torch.full((rows, n_out), float("nan"), dtype=dtype, device=DEV), act, tile_rows=64, most_rows=16)
        assert torch.equal(got, want), dtype
