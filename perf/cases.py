"""The work a user of this library has it do, as cases that can be timed and compared.

Sizes are those of the repository's own configurations (`wallx_mi355.workloads`): hidden 2048, a vision-language expert
of 11008 and an action expert of 1024, 16 query / 2 key-value heads of 128, 36 decoder layers, rows of 912 tokens (three
cameras of 256 image tokens, text, 32 action tokens).  A case is one pass through public entry points:

  moe      decoder layers' mixture-of-experts blocks in inference (`moe.SparseMoeBlock`), a denoise step (action
           tokens only) or a prefill (both experts), eager or replayed from a HIP graph
  train    one block forward and backward, all weights training or the action expert alone
  attn     a decoder layer's projections around attention: the packed rotary table, q / k / v with the rotation, and the
           o projection with the residual; forward, or forward and backward of the first
  rope     the rotary embedding of q and k as an op of its own, forward, or forward and backward
  permute  the token permute / unpermute ops, forward and backward
  index    what a forward builds before its first layer: position ids, the vision tower's rotary table and its window
           permutation, the language model's rotary table
"""

import os
import sys
from types import SimpleNamespace

import torch

sys.path.insert(0, os.path.abspath("wall-x_amd"))  # the package of the tree this runs in

from wallx_mi355 import moe, native, workloads as wl  # noqa: E402
from wallx_mi355.fusions import ops  # noqa: E402

HIDDEN, INTER = wl.HIDDEN, (wl.INTER_VL, wl.INTER_ACT)
HEADS, KV_HEADS, HEAD_DIM = wl.N_Q_HEADS, wl.N_KV_HEADS, wl.HEAD_DIM
QKV = (HEADS + 2 * KV_HEADS) * HEAD_DIM
LAYERS = 36
EPS = 1e-6
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}


def listed():
    return [
        # one robot's denoise step: the 32 action tokens of its chunk through the blocks of all layers, recorded once
        # into a HIP graph and replayed with the norm and the residual folded in
        dict(name="denoise_1_graph", kind="moe", rows=1, row_len=32, action=32, layers=LAYERS, fused=True, ranges=True, graph=True),
        # the same for 64 robots (2048 tokens), the block alone, as the drop-in replacement of the reference's block
        dict(name="denoise_64_graph", kind="moe", rows=64, row_len=32, action=32, layers=LAYERS, fused=False, ranges=True, graph=True),
        # a ragged denoise batch called eagerly, without row ranges from the host: launches and host work count
        dict(name="denoise_7_eager", kind="moe", rows=7, row_len=31, action=31, layers=LAYERS, fused=True, ranges=False, graph=False),
        # one robot's prefill: a single row of 912 tokens
        dict(name="prefill_1", kind="moe", rows=1, row_len=912, action=32, layers=4, fused=True, ranges=True, graph=False),
        # a few rows of odd length, hardly any action tokens among them
        dict(name="prefill_5_ragged", kind="moe", rows=5, row_len=823, action=13, layers=4, fused=True, ranges=True, graph=False),
        # the serving batch: 32 rows, 29184 tokens
        dict(name="prefill_32", kind="moe", rows=32, row_len=912, action=32, layers=1, fused=False, ranges=True, graph=False),
        # fine-tuning the action expert with the vision-language expert frozen, a small batch per GPU
        dict(name="train_4_frozen", kind="train", rows=4, row_len=912, action=32, fused=True, frozen=True),
        # training everything on the largest batch
        dict(name="train_32", kind="train", rows=32, row_len=912, action=32, fused=True, frozen=False),
        # the projections of a prefill of 16 rows
        dict(name="attn_16", kind="attn", rows=16, row_len=912, layout="hf", grad=False),
        # the rotary op as the model's attention calls it in training: tables, forward and backward
        dict(name="rope_16", kind="rope", rows=16, row_len=896, form="tables", layout="hf", dtype="bf16", grad=True),
        # the permute / unpermute pair under autograd, an odd token count
        dict(name="permute_14593", kind="permute", tokens=14593, experts=2, topk=1, dtype="bf16"),
        # a forward's index builders for 16 rows with three cameras each
        dict(name="index_16", kind="index", rows=16, images=3, side=32, text=80, action=32),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "train", "attn", "rope", "permute", "index"])
    if kind == "decode":  # 1 .. 64 robots, chunks of 10 .. 50 action tokens, at most 2048 tokens
        rows, chunk = _log_int(rng, 1, 64), rng.randint(10, 50)
        rows = min(rows, 2048 // chunk)
        return dict(kind="moe", rows=rows, row_len=chunk, action=chunk, layers=LAYERS, fused=rng.random() < 0.5,
                    ranges=rng.random() < 0.7, graph=rng.random() < 0.6)
    rows, row_len = _log_int(rng, 1, 32), rng.randint(280, 912)
    action = rng.choice([0, rng.randint(1, 12), rng.randint(13, 64)])
    if kind == "prefill":
        return dict(kind="moe", rows=rows, row_len=row_len, action=action, layers=4 if rows * row_len <= 8192 else 1,
                    fused=rng.random() < 0.6, ranges=rng.random() < 0.6, graph=False)
    if kind == "train":
        return dict(kind="train", rows=rows, row_len=row_len, action=max(action, 1), fused=rng.random() < 0.7,
                    frozen=rng.random() < 0.4)
    if kind == "attn":
        if rng.random() < 0.4:  # the projections of a denoise step
            row_len = rng.randint(10, 50)
        return dict(kind="attn", rows=rows, row_len=row_len, layout=rng.choice(["hf", "csrc"]), grad=rng.random() < 0.4)
    if kind == "rope":
        form = rng.choice(["tables", "positions", "packed"])
        return dict(kind="rope", rows=rows, row_len=row_len, form=form, layout=rng.choice(["hf", "csrc"]),
                    dtype="bf16" if form == "packed" else rng.choice(["bf16", "bf16", "fp16", "fp32"]),
                    grad=rng.random() < 0.5)
    if kind == "permute":
        topk = rng.choice([1, 1, 2, 3])
        return dict(kind="permute", tokens=_log_int(rng, 100, 29184 // topk), experts=rng.choice([2, 2, 3, 8]), topk=topk,
                    dtype=rng.choice(["bf16", "bf16", "fp16", "fp32"]))
    return dict(kind="index", rows=rows, images=rng.randint(1, 4), side=rng.choice([16, 22, 26, 32, 40]),
                text=rng.randint(8, 120), action=rng.choice([10, 32, 50]))


# ------------------------------------------------------------------------------------------------ shared pieces
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(shape, g, std=1.0, dtype=torch.bfloat16, mean=0.0):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(mean, std, generator=g)


def _token_ids(case, g):
    """[rows, row_len] token ids with `action` action tokens per row at random places (anything else is text)."""
    ids = torch.full((case["rows"], case["row_len"]), wl.TEXT_TOKEN_ID, dtype=torch.int64, device="cuda")
    if case["action"]:
        order = torch.rand(ids.shape, device="cuda", generator=g).argsort(1)[:, :case["action"]]
        ids.scatter_(1, order, wl.ACTION_TOKEN_ID)
    return ids


def _row_counts(case):
    n_action = case["rows"] * case["action"]
    return case["rows"] * case["row_len"] - n_action, n_action


def _row_ranges(case):
    """The CPU tensors of per-expert row ranges that the reference's decoder hands to its blocks."""
    n_vl, n_action = _row_counts(case)
    return torch.tensor([0, n_vl]), torch.tensor([n_vl, n_vl + n_action])


def _block(g):
    """A dual-expert block with random weights of the trained scale, built on the GPU."""
    config = SimpleNamespace(experts=[dict(hidden_size=HIDDEN, intermediate_size=i, hidden_act="silu") for i in INTER])
    with torch.device("meta"):
        block = moe.SparseMoeBlock(config, 2)
    block = block.to(torch.bfloat16).to_empty(device="cuda")
    with torch.no_grad():
        for p in block.parameters():
            p.normal_(0.0, 0.02, generator=g)
    return block


def _positions(rows, row_len, g):
    """[3, rows, row_len] position ids that differ between the axes, as image tokens' do."""
    t = torch.arange(row_len, device="cuda").expand(rows, row_len)
    spread = torch.randint(0, 32, (2, rows, row_len), device="cuda", generator=g)
    return torch.stack([t, t + spread[0], t + spread[1]]).contiguous()


def _leaf(t):
    return t.requires_grad_()


# ------------------------------------------------------------------------------------------------ moe
def _prepare_moe(case, seed):
    g = _gen(seed)
    with torch.no_grad():
        blocks = [_block(g).pack_for_inference() for _ in range(case["layers"])]
    s = SimpleNamespace(case=case, blocks=blocks, ids=_token_ids(case, g), ranges=_row_ranges(case) if case["ranges"] else (None, None))
    shape = (case["rows"], case["row_len"], HIDDEN)
    # the block alone reads hidden states that attention has just written: a few tensors in turn stand for them
    s.h = [_normal(shape, g) for _ in range(1 if case["fused"] else min(4, case["layers"]))]
    s.norms = [_normal((HIDDEN,), g, 0.1, mean=1.0) for _ in range(case["layers"])] if case["fused"] else None
    if case["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _moe_layers(s)
        torch.cuda.current_stream().wait_stream(side)
        s.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s.graph):
            s.out = _moe_layers(s)
    return s


def _moe_layers(s):
    with torch.no_grad():
        types = s.ids == wl.ACTION_TOKEN_ID
        if s.norms is None:
            return [b(s.h[i % len(s.h)], types, *s.ranges) for i, b in enumerate(s.blocks)]
        h = s.h[0]
        for b, w in zip(s.blocks, s.norms):
            h = b(h, types, *s.ranges, pre_norm=(w, EPS), residual=True)
        return h


def _run_moe(s):
    if s.case["graph"]:
        s.graph.replay()
        return s.out
    return _moe_layers(s)


# ------------------------------------------------------------------------------------------------ train
def _prepare_train(case, seed):
    g = _gen(seed)
    block = _block(g)
    if case["frozen"]:
        block.experts[0].requires_grad_(False)
    s = SimpleNamespace(case=case, block=block, ids=_token_ids(case, g))
    s.ranges = _row_ranges(case)
    shape = (case["rows"], case["row_len"], HIDDEN)
    s.h, s.dy = _leaf(_normal(shape, g)), _normal(shape, g, 0.02)
    s.norm = _leaf(_normal((HIDDEN,), g, 0.1, mean=1.0)) if case["fused"] else None
    s.wanted = [s.h] + ([s.norm] if case["fused"] else []) + [p for p in block.parameters() if p.requires_grad]
    return s


def _run_train(s):
    types = s.ids == wl.ACTION_TOKEN_ID
    pre_norm = None if s.norm is None else (s.norm, EPS)
    y = s.block(s.h, types, *s.ranges, pre_norm=pre_norm, residual=s.norm is not None)
    return [y.detach(), *torch.autograd.grad(y, s.wanted, s.dy)]


# ------------------------------------------------------------------------------------------------ attn
def _prepare_attn(case, seed):
    g = _gen(seed)
    rows, row_len, grad = case["rows"], case["row_len"], case["grad"]
    shape = (rows, row_len, HIDDEN)
    s = SimpleNamespace(case=case, pos=_positions(rows, row_len, g), inv_freq=wl.text_inv_freq(HEAD_DIM).cuda())
    s.h, s.residual = _normal(shape, g), _normal(shape, g)
    s.w, s.b, s.wo = _normal((QKV, HIDDEN), g, 0.02), _normal((QKV,), g, 0.02), _normal((HIDDEN, HEADS * HEAD_DIM), g, 0.02)
    s.a = _normal((rows * row_len, HEADS * HEAD_DIM), g)  # what attention would return
    # operands of the row-major dual GEMM's empty second problem
    s.none = (s.a.new_empty(0, HEADS * HEAD_DIM), s.a.new_empty(8, HEADS * HEAD_DIM), s.a.new_empty(0, 8))
    if grad:
        s.wanted = [_leaf(s.h), _leaf(s.w), _leaf(s.b)]
        s.grads = [_normal((rows, n, row_len, HEAD_DIM), g, 0.02) for n in (HEADS, KV_HEADS, KV_HEADS)]
    return s


def _run_attn(s):
    c = s.case
    table = ops.multimodal_rope_table(s.pos, s.inv_freq, wl.MROPE_SECTION, layout=c["layout"])
    q, k, v = ops.qkv_projection_with_rope(s.h, s.w, s.b, table, HEADS, KV_HEADS, mrope_section=wl.MROPE_SECTION,
                                           layout=c["layout"])
    if c["grad"]:
        return [q.detach(), k.detach(), v.detach(), *torch.autograd.grad((q, k, v), s.wanted, s.grads)]
    residual = s.residual.view(-1, HIDDEN)
    out = torch.empty_like(residual)
    native.asym_dual_gmm(s.a, s.none[0], s.wo, s.none[1], out, s.none[2], False, True, add_expert0=residual)
    return [q, k, v, out]


# ------------------------------------------------------------------------------------------------ rope
def _prepare_rope(case, seed):
    g = _gen(seed)
    rows, row_len, dtype = case["rows"], case["row_len"], DTYPES[case["dtype"]]
    s = SimpleNamespace(case=case, pos=_positions(rows, row_len, g), inv_freq=wl.text_inv_freq(HEAD_DIM).cuda())
    # the projections' [rows, row_len, heads, 128] memory behind [rows, heads, row_len, 128] views
    s.q, s.k = (_normal((rows, row_len, n, HEAD_DIM), g, dtype=dtype).transpose(1, 2) for n in (HEADS, KV_HEADS))
    if case["form"] == "tables":  # built once per forward by the model, shared by its layers
        angle = s.pos.float()[..., None] * s.inv_freq
        angle = torch.cat((angle, angle), -1)
        s.tables = (angle.cos().to(dtype), angle.sin().to(dtype))
    elif case["form"] == "packed":
        s.tables = ops.multimodal_rope_table(s.pos, s.inv_freq, wl.MROPE_SECTION, layout=case["layout"])
    if case["grad"]:
        _leaf(s.q), _leaf(s.k)
        s.grads = [_normal((rows, n, row_len, HEAD_DIM), g, dtype=dtype) for n in (HEADS, KV_HEADS)]
    return s


def _run_rope(s):
    c, section = s.case, list(wl.MROPE_SECTION)
    if c["form"] == "tables":
        q, k = ops.multimodal_rope(s.q, s.k, *s.tables, section, layout=c["layout"])
    elif c["form"] == "positions":
        q, k = ops.multimodal_rope_from_positions(s.q, s.k, s.pos, s.inv_freq, section, layout=c["layout"])
    else:
        q, k = ops.multimodal_rope_from_table(s.q, s.k, s.tables, section, layout=c["layout"])
    if c["grad"]:
        return [q.detach(), k.detach(), *torch.autograd.grad((q, k), (s.q, s.k), s.grads)]
    return [q, k]


# ------------------------------------------------------------------------------------------------ permute
def _prepare_permute(case, seed):
    g = _gen(seed)
    T, K, E, dtype = case["tokens"], case["topk"], case["experts"], DTYPES[case["dtype"]]
    s = SimpleNamespace(case=case)
    # each token's K distinct experts, skewed towards the first like the modality split is
    weight = torch.ones(E, device="cuda")
    weight[0] = 8.0
    s.ids = torch.multinomial(weight.expand(T, E), K, generator=g).to(torch.int32)
    s.x, s.dy = _leaf(_normal((T, HIDDEN), g, dtype=dtype)), _normal((T, HIDDEN), g, dtype=dtype)
    s.probs = _leaf(torch.rand((T, K), device="cuda", generator=g).softmax(1)) if K > 1 else None
    return s


def _run_permute(s):
    permuted, row_id_map = ops.permute(s.x, s.ids)
    y = ops.unpermute(permuted, row_id_map, s.probs)
    wanted = (s.x,) if s.probs is None else (s.x, s.probs)
    return [permuted.detach(), row_id_map, y.detach(), *torch.autograd.grad(y, wanted, s.dy)]


# ------------------------------------------------------------------------------------------------ index
def _prepare_index(case, seed):
    g = torch.Generator().manual_seed(seed)
    side, rows, images = case["side"], case["rows"], case["images"]
    n_image = (side // 2) ** 2
    width = case["text"] + case["action"] + images * (n_image + 2) + 10
    ids = torch.full((rows, width), wl.TEXT_TOKEN_ID, dtype=torch.int64)
    for r in range(rows):  # text of varying length in front of the cameras
        at = int(torch.randint(0, case["text"] + 1, (1,), generator=g))
        for _ in range(images):
            ids[r, at] = wl.VISION_START_TOKEN_ID
            ids[r, at + 1:at + 1 + n_image] = wl.IMAGE_TOKEN_ID
            ids[r, at + 1 + n_image] = wl.VISION_END_TOKEN_ID
            at += n_image + 2
        ids[r, width - case["action"]:] = wl.ACTION_TOKEN_ID
    grid = torch.tensor([[1, side, side]] * (rows * images), dtype=torch.int64)
    pad = torch.randint(0, 8, (rows, 1), generator=g)  # left padding
    mask = (torch.arange(width)[None] >= torch.minimum(pad, (ids != wl.TEXT_TOKEN_ID).int().argmax(1, keepdim=True))).to(torch.int64)
    return SimpleNamespace(case=case, ids=ids.cuda(), mask=mask.cuda(), grid=grid.cuda(), grid32=grid.to(torch.int32).cuda(), grid_host=grid,
                           vision_freq=wl.vision_inv_freq().cuda(), text_freq=wl.text_inv_freq(HEAD_DIM).cuda())


def _run_index(s):
    pos, deltas = ops.get_rope_index(s.ids, 2, wl.IMAGE_TOKEN_ID, wl.VIDEO_TOKEN_ID, wl.VISION_START_TOKEN_ID, 2,
                                     image_grid_thw=s.grid, attention_mask=s.mask)
    table = ops.multimodal_rope_table(pos, s.text_freq, wl.MROPE_SECTION)
    vision = ops.rot_pos_emb(s.vision_freq, s.grid, 2, grid_thw_host=s.grid_host)
    window, cu = ops.get_window_index(s.grid32, 112, 2, 14, 4, grid_thw_host=s.grid_host)
    return [pos, deltas, table, vision, window, cu]


# ------------------------------------------------------------------------------------------------ the file's interface
def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(state):
    return globals()["_run_" + state.case["kind"]](state)


def work(case):
    kind = case["kind"]
    if kind in ("moe", "train"):
        counts = _row_counts(case)
        tokens = sum(counts)
        layers = case.get("layers", 1)
        weights = [3 * HIDDEN * i * 2 for i in INTER]
        rows_flops = [6.0 * HIDDEN * i * n for i, n in zip(INTER, counts)]
        live = sum(w for w, n in zip(weights, counts) if n)
        act = tokens * HIDDEN * 2
        if kind == "moe":
            return {"bytes": layers * (live + 2 * act), "flops": layers * sum(rows_flops)}
        # forward, input gradients and the gradients of the weights that train; weights read twice, gradients written once
        trained = weights[1] + (0 if case["frozen"] else weights[0])
        flops = 2 * sum(rows_flops) + rows_flops[1] + (0 if case["frozen"] else rows_flops[0])
        return {"bytes": 2 * live + trained + 4 * act, "flops": flops}
    if kind == "index":
        n_image = case["rows"] * case["images"]
        width = case["text"] + case["action"] + case["images"] * ((case["side"] // 2) ** 2 + 2) + 10
        tokens, patches = case["rows"] * width, n_image * case["side"] ** 2
        return {"bytes": tokens * (8 + 8 + 24 + 4 * HEAD_DIM // 2) + patches * 2 * 20 * 4 + patches // 4 * 4, "flops": 0}
    if kind == "permute":
        T, K, b = case["tokens"], case["topk"], BYTES[case["dtype"]]
        row = HIDDEN * b
        # permute: T rows in, T K out; unpermute: T K in, T out; its backward reads dy (and the rows, for the probabilities'
        # gradient) and writes T K rows; the permute's backward reads those and writes T
        return {"bytes": row * T * (4 + (4 if K == 1 else 5) * K) + 4 * T * K * 3, "flops": 0}
    tokens = case["rows"] * case["row_len"]
    if kind == "rope":
        b = BYTES[case["dtype"]]
        table = {"tables": 2 * HEAD_DIM * b, "positions": 24, "packed": 4 * HEAD_DIM // (2 if case["layout"] == "hf" else 1)}[case["form"]]
        one = tokens * (2 * (HEADS + KV_HEADS) * HEAD_DIM * b + table)
        return {"bytes": one * (2 if case["grad"] else 1), "flops": 0}
    table = tokens * 4 * HEAD_DIM // (2 if case["layout"] == "hf" else 1)
    qkv_flops, o_flops = 2.0 * tokens * HIDDEN * QKV, 2.0 * tokens * HIDDEN * HEADS * HEAD_DIM
    qkv_bytes = 2 * (tokens * (HIDDEN + QKV) + HIDDEN * QKV)
    if case["grad"]:
        return {"bytes": table + 2 * qkv_bytes + 2 * HIDDEN * QKV, "flops": 3 * qkv_flops}
    return {"bytes": table + qkv_bytes + 2 * (3 * tokens * HIDDEN + HIDDEN * HIDDEN), "flops": qkv_flops + o_flops}


def tolerance(case):
    """Each about four times the distance (2-norm) of the path from the same expression in 64 bits without roundings
    in between; the distances measured on an MI355X are given beside it."""
    kind = case["kind"]
    if kind == "index":
        return "exact"
    if kind == "moe":
        # one block 3.9e-3; the residual stream after 4 blocks 8.6e-3, after 36 blocks 1.7e-2 (where a second correct
        # evaluation with eager roundings is 1.7e-2 away as well)
        return {"rel": 3e-2 if case["fused"] else 1.6e-2}
    if kind == "train":  # 3.3e-3 .. 5.5e-3
        return {"rel": 2e-2}
    if kind == "attn":  # 1.7e-3 .. 2.9e-3
        return {"rel": 1e-2}
    # rope: 2.4e-3 in bf16; permute with weights: 2.3e-3 in bf16, 2.8e-4 in fp16, 1.2e-7 in fp32 (cos and sin of angles up
    # to a thousand, evaluated in fp32, add to that in the rope)
    return {"rel": {"bf16": 1e-2, "fp16": 1.2e-3, "fp32": 1e-5}[case["dtype"]]}
