"""Performance cases of the FragPack hot path: what a serving program does with it.

Kinds of case (``case["kind"]``):

- ``decode``: one decode step's attention over compressed records, a few layers
  of a model in a row (the first layer plans the step, the others reuse the
  plan), through ``decode_attention``;
- ``prefill``: causal attention of new tokens over the BF16 workspace, through
  ``flash_attn_varlen_func`` (fresh prompts, chunks over a context, the short
  remainder of a chunked prompt);
- ``store``: the new tokens of a step stored, every completed block encoded and
  read back token-major, through ``HbmKvStore`` (prepare, per layer write +
  encode, commit, gather);
- ``blobs``: closed blocks exported to blobs and installed into other blocks
  (KV offload, prefix sharing);
- ``serve``: a whole engine step through ``FragPackRunner`` (build, then
  ``layer_forward`` per layer): decode rows over long contexts and, with
  ``chunk``, a prefill chunk in the same step.

K and V are N(0, 1) times a per-channel lognormal(0, 0.5) scale with a few
outlier channels x8 (``heavy``: a tenth of the values from a Student-t(2) x 16
tail, which records cannot code); tables are calibrated on such data; queries
are N(0, 1); everything is BF16 with head size 128.
"""

from __future__ import annotations

import math

import numpy as np
import torch

T = 128  # tokens of a block
D = 128  # head size
SCALE = D ** -0.5
DENSE = 22528
CODED = DENSE + 576  # typical bytes of a coded record of this data
RAW = 32768


def listed() -> list[dict]:
    return [
        # One user, a short chat: the smallest decode (7 closed blocks and a raw tail), all latency.
        dict(name="decode_1x1000", kind="decode", heads=4, group=8, layers=4, lens="1000", outlier=0.02),
        # A small batch of 8K contexts on a GQA-8 model.
        dict(name="decode_4x8192", kind="decode", heads=4, group=8, layers=8, lens="8192x4", outlier=0.02),
        # MHA (no grouping), ragged contexts with raw tails.
        dict(name="decode_mha_ragged", kind="decode", heads=32, group=1, layers=1,
             lens="2113,3987,129,1540,777,4096,2901,350,3333,1024,1871,2500,600,3701,1290,2222", outlier=0.05),
        # Throughput serving of long contexts: the largest decode.
        dict(name="decode_64x32768", kind="decode", heads=8, group=4, layers=1, lens="32768x64", outlier=0.02),
        # Four long prompts prefilled whole.
        dict(name="prefill_4x8192", kind="prefill", heads=8, group=4, q="8192x4", ctx="0x4"),
        # Fresh prompts of everyday lengths in one step.
        dict(name="prefill_ragged", kind="prefill", heads=8, group=4, q="1000,37,2311,512", ctx="0x4"),
        # A chunk of four long prompts over what is already there.
        dict(name="prefill_chunk", kind="prefill", heads=8, group=4, q="1024x4", ctx="8192x4"),
        # The last, short chunk of a long prompt.
        dict(name="prefill_tail", kind="prefill", heads=4, group=8, q="200", ctx="8192"),
        # A step of four long prompts stored and read back, four layers.
        dict(name="store_32768", kind="store", heads=8, layers=4, tokens=32768, outlier=0.02, heavy=False),
        # The same path for one chunk whose values often do not code.
        dict(name="store_8192_heavy", kind="store", heads=8, layers=1, tokens=8192, outlier=0.02, heavy=True),
        # Offload and reload of 64 blocks of four layers.
        dict(name="blobs_64x4", kind="blobs", heads=8, layers=4, blocks=64, outlier=0.02),
        # An engine step: 16 decodes beside a 1024-token chunk of a prompt, two layers.
        dict(name="serve_mixed", kind="serve", heads=8, group=4, layers=2, lens="4001x16", chunk=1024, chunk_ctx=2048,
             outlier=0.02),
    ]


def draw(rng) -> dict:
    def log(lo: float, hi: float) -> int:
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["decode", "decode", "prefill", "prefill", "store", "blobs", "serve"])
    heads = rng.choice([4, 8, 8, 16, 32])
    group = rng.choice([1, 2, 4, 8])
    outlier = rng.choice([0.02, 0.05])
    if kind == "decode":
        batch, ctx = log(1, 64), log(40, 32768)
        while batch * ctx * heads > 64 * 32768 * 4:
            batch = max(1, batch // 2)
        ragged = rng.random() < 0.6
        lens = [rng.randint(max(1, ctx // 8), ctx) if ragged else ctx for _ in range(batch)]
        layers = rng.choice([1, 2, 4]) if sum(lens) * heads < 1 << 19 else 1
        return dict(kind=kind, heads=heads, group=group, layers=layers, lens=_text(lens), outlier=outlier)
    if kind == "prefill":
        n, new, ctx = rng.choice([1, 1, 2, 3, 5]), log(16, 6000), rng.choice([0, 0, log(100, 12000)])
        heads = min(heads, 8)
        q = [max(1, rng.randint(new // 4, new)) if rng.random() < 0.7 else new for _ in range(n)]
        return dict(kind=kind, heads=heads, group=min(group, 32 // heads), q=_text(q),
                    ctx=_text([rng.randint(0, ctx) for _ in range(n)]))
    if kind == "store":
        heads = min(heads, 16)
        return dict(kind=kind, heads=heads, layers=rng.choice([1, 2, 4]), tokens=T * log(1, 2048 // heads),
                    outlier=outlier, heavy=rng.random() < 0.25)
    if kind == "blobs":
        heads = min(heads, 16)
        return dict(kind=kind, heads=heads, layers=rng.choice([1, 2, 4]), blocks=log(1, 512 // heads), outlier=outlier)
    heads = min(heads, 8)
    lens = [rng.randint(130, 6000) // T * T + rng.randint(1, 127) for _ in range(log(1, 48))]
    chunk = rng.choice([0, T * log(1, 16)])
    return dict(kind="serve", heads=heads, group=group, layers=rng.choice([1, 2]), lens=_text(lens), chunk=chunk,
                chunk_ctx=T * rng.randint(0, 40), outlier=outlier)


def _text(values: list[int]) -> str:
    return ",".join(str(v) for v in values)


def _ints(text: str) -> list[int]:
    """"a,bxn,.." -> [a, b (n times), ..]"""
    out: list[int] = []
    for part in text.split(","):
        v, _, n = part.partition("x")
        out += [int(v)] * int(n or 1)
    return out


def _pages(n: int) -> int:
    return -(-n // T)


# ---------------------------------------------------------------------------
# Inputs, from the seed alone.


def _gen(seed: int, *stream: int) -> torch.Generator:
    s = seed
    for x in stream:
        s = (s * 1000003 + x + 1) % (1 << 62)
    return torch.Generator(device="cuda").manual_seed(s)


def _normal(gen: torch.Generator, *shape: int) -> torch.Tensor:
    return torch.randn(shape, generator=gen, device="cuda")


def _channel_scales(seed: int, heads: int, outlier: float) -> torch.Tensor:
    """[2, H, 128]"""
    gen = _gen(seed, 11)
    s = torch.exp(0.5 * _normal(gen, 2, heads, D))
    out = torch.rand((2, heads, D), generator=gen, device="cuda") < outlier
    return torch.where(out, 8 * s, s)


def _kv(gen: torch.Generator, scales: torch.Tensor, tokens: int, heavy: bool = False) -> torch.Tensor:
    """BF16 [2, tokens, H, 128]"""
    heads = scales.shape[1]
    x = _normal(gen, 2, tokens, heads, D).mul_(scales[:, None])
    if heavy:
        chi = _normal(gen, 2, tokens, heads, D).square_() + _normal(gen, 2, tokens, heads, D).square_()
        t2 = _normal(gen, 2, tokens, heads, D) / torch.sqrt(chi / 2) * 16
        x = torch.where(torch.rand(x.shape, generator=gen, device="cuda") < 0.1, t2, x)
    return x.to(torch.bfloat16)


def _queries(seed: int, layer: int, rows: int, heads: int) -> torch.Tensor:
    return _normal(_gen(seed, 12, layer), rows, heads, D).to(torch.bfloat16)


def _tables(seed: int, scales: torch.Tensor, layers: int):
    """Calibrated device tables, the same for every layer."""
    from fragpack_amd.compression.attn_tables import calibrate, device_tables

    dump = _kv(_gen(seed, 13), scales, 4 * T).view(2, 4, T, -1, D).transpose(0, 1).contiguous()  # [4, 2, T, H, D]
    tables = calibrate(dump.view(torch.int16).cpu().numpy().view(np.uint16)[:, None])
    return device_tables(np.repeat(tables, layers, axis=0), torch.device("cuda"))


class _Contexts:
    """Sequences' past KV: block ids (scattered over the cache), and the
    token-major K / V by page, drawn a stretch of pages at a time."""

    STRETCH = 1024

    def __init__(self, seed: int, lens: list[int], heads: int, outlier: float, spare: int = 0) -> None:
        self.seed, self.lens, self.heads = seed, lens, heads
        self.scales = _channel_scales(seed, heads, outlier)
        self.pages = [_pages(n) for n in lens]
        self.total = sum(self.pages)
        self.first = [sum(self.pages[:i]) for i in range(len(lens))]
        self.num_blocks = self.total + spare
        self.blocks = np.random.default_rng(seed).permutation(self.num_blocks).astype(np.int64)
        # tokens held by each page
        self.held = np.concatenate([np.minimum(T, n - T * np.arange(_pages(n))) for n in lens] or [np.zeros(0)])

    def stretches(self, layer: int):
        """(first page, BF16 K/V [2, pages * 128, H, 128]) in page order"""
        for p0 in range(0, self.total, self.STRETCH):
            n = min(self.STRETCH, self.total - p0)
            yield p0, _kv(_gen(self.seed, 14, layer, p0), self.scales, n * T)

    def kv(self, layer: int) -> torch.Tensor:
        """BF16 [2, pages, 128, H, 128]"""
        out = torch.empty((2, self.total, T, self.heads, D), dtype=torch.bfloat16, device="cuda")
        for p0, kv in self.stretches(layer):
            n = kv.shape[1] // T
            out[:, p0 : p0 + n] = kv.view(2, n, T, self.heads, D)
        return out

    def fill(self, store, layers: int) -> np.ndarray:
        """Store every sequence's tokens, as steps of an engine; returns the
        blocks left open (partly filled: raw in staging)."""
        live = np.zeros(0, np.int32)
        gens = [self.stretches(layer) for layer in range(layers)]
        for p0 in range(0, self.total, self.STRETCH):
            n = min(self.STRETCH, self.total - p0)
            held, blocks = self.held[p0 : p0 + n], self.blocks[p0 : p0 + n]
            keep = np.arange(T)[None, :] < held[:, None]
            slots = torch.from_numpy((blocks[:, None] * T + np.arange(T)[None, :])[keep]).cuda()
            rows = None if keep.all() else torch.from_numpy(np.flatnonzero(keep)).cuda()
            store.prepare(slots, slots.numel(), live)
            for layer in range(layers):
                _, kv = next(gens[layer])
                if rows is not None:
                    kv = kv[:, rows]
                store.write(layer, kv[0], kv[1], slots)
                store.encode(layer, n)
            store.commit()
            live = np.concatenate((live, blocks[held < T])).astype(np.int32)
        return live

    def block_table(self) -> torch.Tensor:
        bt = np.zeros((len(self.lens), max(1, max(self.pages))), np.int32)
        for b, (f, n) in enumerate(zip(self.first, self.pages)):
            bt[b, :n] = self.blocks[f : f + n]
        return torch.from_numpy(bt).cuda()


def _caches(layers: int, blocks: int, heads: int) -> list[torch.Tensor]:
    from fragpack_amd.ops.hbm_kv import page_bytes

    return [torch.empty((blocks, page_bytes(heads)), dtype=torch.uint8, device="cuda") for _ in range(layers)]


def _decode_workspace(batch: int, heads: int):
    from fragpack_amd.ops.fused_attn_decode import decode_units, workspace_elems

    cus = torch.cuda.get_device_properties(torch.device("cuda")).multi_processor_count
    units = decode_units(batch, heads, cus)
    opart, ml, plan = workspace_elems(heads, units)
    return units, (torch.empty(opart, dtype=torch.float32, device="cuda"),
                   torch.empty(ml, dtype=torch.float32, device="cuda"),
                   torch.zeros(plan, dtype=torch.int32, device="cuda"))


# ---------------------------------------------------------------------------
# prepare / run


def prepare(case: dict, seed: int):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_decode(case: dict, seed: int):
    from fragpack_amd.ops.fused_attn_decode import RecordTables
    from fragpack_amd.ops.hbm_kv import HbmKvStore

    lens, heads, layers = _ints(case["lens"]), case["heads"], case["layers"]
    ctx = _Contexts(seed, lens, heads, case["outlier"])
    caches = _caches(layers, ctx.num_blocks, heads)
    store = HbmKvStore(caches, heads, _tables(seed, ctx.scales, layers),
                       max_tokens=min(ctx.total, ctx.STRETCH) * T, staging_slots=len(lens), overflow_records=1024)
    ctx.fill(store, layers)
    q = [_queries(seed, i, len(lens), heads * case["group"]) for i in range(layers)]
    units, workspace = _decode_workspace(len(lens), heads)
    return dict(run=_run_decode, store=store, caches=caches, q=q, out=[torch.empty_like(x) for x in q],
                tables=[RecordTables(*store.layer_tables(i)) for i in range(layers)], block_table=ctx.block_table(),
                lens=torch.tensor(lens, dtype=torch.int32, device="cuda"), units=units, workspace=workspace)


def _run_decode(s):
    from fragpack_amd.ops.fused_attn_decode import decode_attention

    for i, q in enumerate(s["q"]):
        decode_attention(q, s["tables"][i], s["block_table"], s["lens"], SCALE, s["units"], s["out"][i],
                         s["workspace"], replan=i == 0)
    return s["out"]


def _prefill_inputs(case: dict, seed: int):
    nq, past, heads = _ints(case["q"]), _ints(case["ctx"]), case["heads"]
    ctx = _Contexts(seed, [a + b for a, b in zip(nq, past)], heads, 0.02)
    kv = ctx.kv(0)
    return nq, ctx, kv, _queries(seed, 0, sum(nq), heads * case["group"])


def _prepare_prefill(case: dict, seed: int):
    nq, ctx, kv, q = _prefill_inputs(case, seed)
    bt = np.zeros((len(nq), max(ctx.pages)), np.int32)
    for b, (f, n) in enumerate(zip(ctx.first, ctx.pages)):
        bt[b, :n] = np.arange(f, f + n)  # the workspace holds a group's pages in order
    i32 = dict(dtype=torch.int32, device="cuda")
    return dict(run=_run_prefill, q=q, k=kv[0].contiguous(), v=kv[1].contiguous(), out=torch.empty_like(q),
                cu_q=torch.tensor(np.concatenate(([0], np.cumsum(nq))), **i32), used_k=torch.tensor(ctx.lens, **i32),
                block_table=torch.from_numpy(bt).cuda(), max_q=max(nq), max_k=max(ctx.lens))


def _run_prefill(s):
    from fragpack_amd.ops.prefill_attn import flash_attn_varlen_func

    return flash_attn_varlen_func(q=s["q"], k=s["k"], v=s["v"], out=s["out"], cu_seqlens_q=s["cu_q"],
                                  max_seqlen_q=s["max_q"], seqused_k=s["used_k"], max_seqlen_k=s["max_k"],
                                  softmax_scale=SCALE, causal=True, block_table=s["block_table"])


def _store_kv(case: dict, seed: int, scales: torch.Tensor) -> list[torch.Tensor]:
    return [_kv(_gen(seed, 15, i), scales, case["tokens"], case["heavy"]) for i in range(case["layers"])]


def _prepare_store(case: dict, seed: int):
    from fragpack_amd.ops.hbm_kv import HbmKvStore

    heads, layers, tokens = case["heads"], case["layers"], case["tokens"]
    n = tokens // T
    scales = _channel_scales(seed, heads, case["outlier"])
    caches = _caches(layers, 2 * n, heads)
    store = HbmKvStore(caches, heads, _tables(seed, scales, layers), max_tokens=tokens, staging_slots=8,
                       overflow_records=2 * heads * n * layers if case["heavy"] else 1024)
    blocks = np.random.default_rng(seed).permutation(2 * n)[:n].astype(np.int64)
    kv = _store_kv(case, seed, scales)
    pages = lambda: [torch.empty((n, T, heads, D), dtype=torch.bfloat16, device="cuda") for _ in range(layers)]  # noqa: E731
    return dict(run=_run_store, store=store, caches=caches, blocks=torch.from_numpy(blocks.astype(np.int32)).cuda(),
                slots=torch.from_numpy((blocks[:, None] * T + np.arange(T)).reshape(-1)).cuda(), kv=kv, wk=pages(),
                wv=pages(), live=np.zeros(0, np.int32))


def _run_store(s):
    store, slots, n = s["store"], s["slots"], s["blocks"].numel()
    store.prepare(slots, slots.numel(), s["live"])
    for i, kv in enumerate(s["kv"]):
        if slots.numel() <= 512:
            store.write_encode(i, kv[0], kv[1], slots, n)
        else:
            store.write(i, kv[0], kv[1], slots)
            store.encode(i, n)
    store.commit()
    for i in range(len(s["kv"])):
        store.gather(i, s["blocks"], s["wk"][i], s["wv"][i])
    return [*s["wk"], *s["wv"]]


def _prepare_blobs(case: dict, seed: int):
    from fragpack_amd.ops.hbm_kv import HbmKvStore

    heads, layers, n = case["heads"], case["layers"], case["blocks"]
    ctx = _Contexts(seed, [T] * n, heads, case["outlier"], spare=n)
    caches = _caches(layers, ctx.num_blocks, heads)
    store = HbmKvStore(caches, heads, _tables(seed, ctx.scales, layers), max_tokens=min(ctx.total, ctx.STRETCH) * T,
                       staging_slots=8, overflow_records=1024)
    ctx.fill(store, layers)
    ids = torch.from_numpy(ctx.blocks.astype(np.int32)).cuda()
    stride = store.blob_stride
    return dict(run=_run_blobs, store=store, caches=caches, src=ids[:n].contiguous(), dst=ids[n:].contiguous(),
                blobs=torch.zeros(n * stride, dtype=torch.uint8, device="cuda"), stride=stride,
                offsets=torch.arange(n, dtype=torch.int64, device="cuda") * stride,
                pages=[torch.empty((n, T, heads, D), dtype=torch.bfloat16, device="cuda") for _ in range(2 * layers)])


def _run_blobs(s):
    store, pages = s["store"], s["pages"]
    lengths = store.export_blocks(s["src"], s["blobs"], s["stride"])
    status = store.import_blocks(s["blobs"], s["offsets"], s["dst"])
    for i in range(len(pages) // 2):
        store.gather(i, s["dst"], pages[2 * i], pages[2 * i + 1])
    return [s["blobs"], lengths, status, *pages]


def _serve_inputs(case: dict, seed: int):
    """Contexts before the step (decode rows: all but the new token; then the
    chunk's sequence), the step's query lengths and its new K / V."""
    heads, lens, chunk = case["heads"], _ints(case["lens"]), case["chunk"]
    seqs = lens + ([case["chunk_ctx"] + chunk] if chunk else [])
    nq = [1] * len(lens) + ([chunk] if chunk else [])
    past = _Contexts(seed, [n - k for n, k in zip(seqs, nq)], heads, case["outlier"],
                     spare=len(lens) + _pages(chunk))
    new = [_kv(_gen(seed, 16, i), past.scales, sum(nq)) for i in range(case["layers"])]
    return seqs, nq, past, new


def _prepare_serve(case: dict, seed: int):
    from fragpack_amd.integrations.vllm.step import FragPackRunner

    heads, layers = case["heads"], case["layers"]
    seqs, nq, past, new = _serve_inputs(case, seed)
    rows = len(seqs)
    caches = _caches(layers, past.num_blocks, heads)
    runner = FragPackRunner(heads, _tables(seed, past.scales, layers), "cuda",
                            max_tokens=max(min(past.total, past.STRETCH) * T, sum(nq)), max_reqs=rows,
                            max_model_len=max(seqs), overflow_records=1024)
    live = past.fill(runner.bind(caches), layers)
    # the sequences' blocks: past pages, then spare ones
    spare = list(past.blocks[past.total :])
    table = np.zeros((rows, max(_pages(n) for n in seqs)), np.int32)
    slots = []
    for b, (n, k) in enumerate(zip(seqs, nq)):
        ids = list(past.blocks[past.first[b] : past.first[b] + past.pages[b]])
        while len(ids) < _pages(n):
            ids.append(spare.pop())
        table[b, : len(ids)] = ids
        pos = np.arange(n - k, n)
        slots.append(np.asarray(ids)[pos // T] * T + pos % T)
    q = [_queries(seed, i, sum(nq), heads * case["group"]) for i in range(layers)]
    return dict(run=_run_serve, runner=runner, caches=caches, q=q, kv=new, out=[torch.empty_like(x) for x in q],
                starts=np.concatenate(([0], np.cumsum(nq))), lens_host=np.asarray(seqs, np.int64),
                lens=torch.tensor(seqs, dtype=torch.int32, device="cuda"), table=torch.from_numpy(table).cuda(),
                slots=torch.from_numpy(np.concatenate(slots).astype(np.int64)).cuda(), live=live)


def _run_serve(s):
    from fragpack_amd.integrations.vllm.step import layer_forward

    md = s["runner"].build(s["caches"], s["starts"], s["lens_host"], s["lens"], s["table"], s["slots"], s["live"])
    for i, kv in enumerate(s["kv"]):
        layer_forward(md, i, s["q"][i], kv[0], kv[1], s["out"][i], SCALE)
    return s["out"]


_PREPARE = {"decode": _prepare_decode, "prefill": _prepare_prefill, "store": _prepare_store, "blobs": _prepare_blobs,
            "serve": _prepare_serve}


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how exact it is.


def _record_bytes(lens: list[int], heads: int) -> int:
    """Bytes of the K and V records of sequences: coded, the open page raw."""
    return sum(2 * heads * (n // T * CODED + (n % T > 0) * RAW) for n in lens)


def _attended(nq: list[int], past: list[int]) -> int:
    """Query-key pairs under the causal mask."""
    return sum(q * p + q * (q + 1) // 2 for q, p in zip(nq, past))


def work(case: dict) -> dict:
    kind, heads, layers = case["kind"], case["heads"], case.get("layers", 1)
    row = 2 * D  # bytes of one head's row
    if kind == "decode":
        lens, hq = _ints(case["lens"]), heads * case["group"]
        return {"bytes": layers * (_record_bytes(lens, heads) + 2 * len(lens) * hq * row),
                "flops": layers * 4 * D * hq * sum(lens)}
    if kind == "prefill":
        nq, past, hq = _ints(case["q"]), _ints(case["ctx"]), heads * case["group"]
        return {"bytes": 2 * sum(nq) * hq * row + 2 * (sum(nq) + sum(past)) * heads * row,
                "flops": 4 * D * hq * _attended(nq, past)}
    if kind == "store":
        # tokens in, records out; records in, tokens out
        n = layers * 2 * heads * (case["tokens"] // T)
        return {"bytes": 2 * n * (RAW + (RAW if case["heavy"] else CODED)), "flops": 0}
    if kind == "blobs":
        # records out to blobs, blobs in to records, records read back token-major
        return {"bytes": layers * 2 * heads * case["blocks"] * (5 * CODED + RAW), "flops": 0}
    lens, hq, chunk, past = _ints(case["lens"]), heads * case["group"], case["chunk"], case["chunk_ctx"]
    tokens = len(lens) + chunk
    moved = _record_bytes(lens, heads) + 2 * tokens * hq * row + 2 * 2 * tokens * heads * row
    if chunk:
        moved += _record_bytes([past + chunk], heads) + 2 * 2 * (past + chunk) * heads * row
    return {"bytes": layers * moved, "flops": layers * 4 * D * hq * (sum(lens) + _attended([chunk], [past]))}


def tolerance(case: dict):
    if case["kind"] in ("store", "blobs"):
        return "exact"  # bytes
    # BF16 output rows and BF16 probabilities, sums in fp32
    return {"rel": 1e-2, "max": 4e-2}


def _attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, past: int) -> torch.Tensor:
    """float64 causal attention of q [n, Hq, 128] at positions past.. over k / v [>= past + n, H, 128]"""
    n, hq = q.shape[:2]
    heads = k.shape[1]
    group = hq // heads
    out = torch.empty((n, hq, D), dtype=torch.float64, device=q.device)
    for h in range(heads):
        kt = k[: past + n, h].double().t().contiguous()
        vh = v[: past + n, h].double().contiguous()
        for g in range(group):
            for r0 in range(0, n, 2048):
                rows = q[r0 : r0 + 2048, h * group + g].double().contiguous()
                end = past + r0 + rows.shape[0]
                s = (rows @ kt[:, :end].contiguous()) * SCALE
                if rows.shape[0] > 1:
                    pos = torch.arange(past + r0, end, device=q.device)
                    s.masked_fill_(torch.arange(end, device=q.device)[None, :] > pos[:, None], -math.inf)
                out[r0 : r0 + 2048, h * group + g] = s.softmax(-1) @ vh[:end]
    return out


def _decode_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
    """float64 attention of q [Hq, 128] over k / v [n, H, 128]"""
    heads = k.shape[1]
    kt = k.double().permute(1, 2, 0).contiguous()
    vt = v.double().transpose(0, 1).contiguous()
    s = torch.bmm(q.double().view(heads, -1, D), kt) * SCALE
    return torch.bmm(s.softmax(-1), vt).reshape(-1, D)


def exact(case: dict, seed: int):
    kind, heads = case["kind"], case["heads"]
    if kind == "decode":
        lens, group = _ints(case["lens"]), case["group"]
        ctx = _Contexts(seed, lens, heads, case["outlier"])
        outs = []
        for layer in range(case["layers"]):
            kv = ctx.kv(layer).view(2, -1, heads, D)
            q = _queries(seed, layer, len(lens), heads * group)
            outs.append(torch.stack([_decode_attention(q[b], kv[0, T * f : T * f + n], kv[1, T * f : T * f + n])
                                     for b, (f, n) in enumerate(zip(ctx.first, lens))]))
        return outs
    if kind == "prefill":
        nq, ctx, kv, q = _prefill_inputs(case, seed)
        kv = kv.view(2, -1, heads, D)
        starts = np.concatenate(([0], np.cumsum(nq)))
        return torch.cat([_attention(q[starts[b] : starts[b + 1]], kv[0, T * f : T * f + n], kv[1, T * f : T * f + n],
                                     n - nq[b]) for b, (f, n) in enumerate(zip(ctx.first, ctx.lens))])
    if kind == "store":
        kv = _store_kv(case, seed, _channel_scales(seed, heads, case["outlier"]))
        pages = [x.view(2, -1, T, heads, D) for x in kv]
        return [*(x[0] for x in pages), *(x[1] for x in pages)]
    if kind == "blobs":
        ctx = _Contexts(seed, [T] * case["blocks"], heads, case["outlier"], spare=case["blocks"])
        return [None, None, None, *(x for layer in range(case["layers"]) for x in ctx.kv(layer))]
    seqs, nq, past, new = _serve_inputs(case, seed)
    starts = np.concatenate(([0], np.cumsum(nq)))
    outs = []
    for layer in range(case["layers"]):
        old = past.kv(layer).view(2, -1, heads, D)
        q = _queries(seed, layer, sum(nq), heads * case["group"])
        rows = []
        for b, (f, n) in enumerate(zip(past.first, seqs)):
            s, e = starts[b], starts[b + 1]
            k, v = (torch.cat((old[i, T * f : T * f + n - nq[b]], new[layer][i, s:e])) for i in (0, 1))
            rows.append(_decode_attention(q[s], k, v)[None] if nq[b] == 1 else _attention(q[s:e], k, v, n - nq[b]))
        outs.append(torch.cat(rows))
    return outs
