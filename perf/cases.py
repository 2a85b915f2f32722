"""What the save/load path of a KV-cache connector is asked to do, as cases that can be timed and compared.

A case is a dict of plain values. `listed()` names twelve that stand for the calls a serving process makes; `draw(rng)`
gives more of the same ranges. `prepare(case, seed)` makes what the caller has in hand before the call, `run(state)` is one
pass through the public entry points, `work(case)` what no implementation can do without, `tolerance(case)` how far two
correct implementations may differ (not at all: everything here is whole numbers and bytes).

Kinds of case:
  keys    block keys of token IDs           hashing.hash_tokens            requests [R, L], or ragged with offsets
  chain   keys over ready block digests     hashing.apply_prefix_hash      ragged sequences
  sha     keys of radix-tree hash strings   hashing.sha256_to_int64        host strings in, device keys out
  select  which blocks of a batch to save   save_selection.select_save_indices
  task    one transfer task of the connector  connector.DataTransferManager.save_task / load_task
  copy    the gather/scatter operators      kernel.batch_gather_scatter_helper, index as "list" (Python list of token
          slots), "slots" (device tensor of token slots) or "table" (device tensor of run starts)
"""
import math
import random

import numpy as np
import torch

from tair_kvcache_amd import client_types, connector, hashing, save_selection
from tair_kvcache_amd.kernel import batch_gather_scatter_helper as bgs
from tair_kvcache_amd.kernel.gather_scatter_helper import CopyBufferAllocator

DEVICE = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "u8": torch.uint8}  # u8: how engines hold an fp8 cache
VOCAB = 128256
MOST_TOKENS = 16384 * 4096
MOST_STAGED_BYTES = 200 * 160 * 64 * 2048


def listed():
    return [
        # A handful of short prompts arrives: launches and host time are all there is.
        {"name": "keys_4x512", "kind": "keys", "requests": 4, "shortest": 512, "longest": 512, "block": 16, "bits": 64},
        # One full prefill batch of equally long prompts at the usual block size.
        {"name": "keys_64x4096", "kind": "keys", "requests": 64, "shortest": 4096, "longest": 4096, "block": 16, "bits": 64},
        # The same as it comes in earnest: prompts of every length, 32-bit token IDs, flat with offsets.
        {"name": "keys_ragged_i32", "kind": "keys", "requests": 160, "shortest": 48, "longest": 8192, "block": 16, "bits": 32},
        # Re-keying a whole trace or a manager's backlog: every compute unit busy, 512 MiB of tokens.
        {"name": "keys_16384x4096", "kind": "keys", "requests": 16384, "shortest": 4096, "longest": 4096, "block": 16,
         "bits": 64},
        # Trace conversion: per-block digests are there already and only have to be chained.
        {"name": "chain_1000", "kind": "chain", "requests": 1000, "shortest": 8, "longest": 1024},
        # A radix-tree engine names its pages by SHA-256 hex strings; one request of 1024 pages.
        {"name": "sha_1024", "kind": "sha", "strings": 1024, "characters": 64},
        # Keys of a batch of 512 requests against each other and the manager's mask: what is left to save.
        {"name": "select_32768", "kind": "select", "requests": 512, "blocks": 64, "saved": 0.4},
        # The connector's save task: 128 blocks of an 8B-class model (32 layers, 8 KV heads x 128), index as the nested
        # lists of the scheduler, staging slot allocation and the wait for the copy included.
        {"name": "task_save_8b", "kind": "task", "save": True, "layers": 32, "kv": 2, "row": 1024, "dtype": "bf16",
         "manager_block": 16, "engine_block": 16, "blocks": 128},
        # A short prefix hit of a 0.5B-class model (24 layers, 2 KV heads x 64) is loaded: 20 blocks, list of slots.
        {"name": "load_small", "kind": "copy", "save": False, "layers": 24, "kv": 2, "row": 128, "dtype": "bf16",
         "manager_block": 16, "engine_block": 16, "blocks": 20, "index": "list"},
        # Long-context load at a 72B-class shape: 80 layers, 64-token blocks, 4 GiB in one call, block table on the device.
        {"name": "load_72b", "kind": "copy", "save": False, "layers": 80, "kv": 2, "row": 1024, "dtype": "bf16",
         "manager_block": 64, "engine_block": 64, "blocks": 200, "index": "table"},
        # Save of a latent-attention cache held in fp8: one 576-byte row per token and layer, 128-token manager blocks over
        # 64-token engine blocks.
        {"name": "save_mla_fp8", "kind": "copy", "save": True, "layers": 61, "kv": 1, "row": 576, "dtype": "u8",
         "manager_block": 128, "engine_block": 64, "blocks": 250, "index": "table"},
        # Page size 1: every token of a block sits somewhere else in the pool (28 layers, 4 KV heads x 128).
        {"name": "load_page1", "kind": "copy", "save": False, "layers": 28, "kv": 2, "row": 512, "dtype": "fp16",
         "manager_block": 16, "engine_block": 1, "blocks": 2000, "index": "slots"},
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _draw_layout(rng, page1):
    if rng.random() < 0.25:  # latent attention: one row per token and layer
        kv, row, dtype = 1, 576, rng.choice(["bf16", "u8"])
    else:  # grouped-query attention, whole or as one rank of a tensor-parallel group holds it
        kv, row, dtype = 2, rng.choice([1, 2, 4, 8]) * rng.choice([64, 80, 128, 128, 256]), rng.choice(["bf16", "fp16", "u8"])
    block = rng.choice([16, 16, 32, 64, 128])
    engine = 1 if page1 else rng.choice([e for e in (8, 16, 32, 64, 128) if e <= block])
    return {"layers": rng.randint(12, 80), "kv": kv, "row": row, "dtype": dtype, "manager_block": block,
            "engine_block": engine}


def draw(rng):
    kind = rng.choice(["keys", "keys", "keys", "chain", "sha", "select", "task", "copy", "copy", "copy", "copy"])
    if kind == "keys":
        block = rng.choice([8, 16, 16, 16, 24, 32, 64, 128])
        longest = _log_int(rng, max(64, 2 * block), 32768)
        shortest = longest if rng.random() < 0.4 else max(1, longest // rng.choice([2, 8, 64]))
        return {"kind": kind, "requests": _log_int(rng, 1, min(16384, MOST_TOKENS // longest)), "shortest": shortest,
                "longest": longest, "block": block, "bits": rng.choice([32, 64])}
    if kind == "chain":
        longest = _log_int(rng, 8, 4096)
        return {"kind": kind, "requests": _log_int(rng, 1, 8192), "shortest": max(1, longest // rng.choice([1, 4, 64])),
                "longest": longest}
    if kind == "sha":
        return {"kind": kind, "strings": _log_int(rng, 1, 16384), "characters": rng.choice([16, 64, 64, rng.randint(1, 200)])}
    if kind == "select":
        blocks = _log_int(rng, 4, 512)
        return {"kind": kind, "requests": _log_int(rng, 1, (1 << 20) // blocks), "blocks": blocks,
                "saved": round(rng.uniform(0.0, 0.9), 2)}
    index = rng.choice(["list", "slots", "table"])
    case = {"kind": kind, "save": rng.random() < 0.5}
    case.update(_draw_layout(rng, kind == "copy" and index == "slots" and rng.random() < 0.7))
    most = MOST_STAGED_BYTES // _block_bytes(case)
    if kind == "task":
        case["blocks"] = _log_int(rng, 1, min(256, most))
        return case
    case["blocks"] = _log_int(rng, 1, min(most, 65536 // case["manager_block"] if index == "list" else 8192))
    case["index"] = index
    return case


# ------------------------------------------------------------------------------------------------ inputs

def _lengths(case, seed):
    """Lengths of the case's requests, spread over their logarithm between the shortest and the longest. They belong to
    the case, the seed only deals them out, so that the work of a case is the same for every seed."""
    low, high, n = case["shortest"], case["longest"], case["requests"]
    spread = np.exp(np.linspace(math.log(low), math.log(high), n)).round().astype(np.int64).clip(low, high)
    return np.random.default_rng(seed).permutation(spread)


def _offsets(lengths):
    return np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)


def _block_bytes(case):
    itemsize = torch.empty(0, dtype=DTYPES[case["dtype"]]).element_size()
    return case["layers"] * case["kv"] * case["manager_block"] * case["row"] * itemsize


def _fill(t, gen):
    """Cache contents: normal values, or bytes over the finite codes of an 8-bit float."""
    if t.dtype == torch.uint8:
        return t.random_(0, 127, generator=gen)
    return t.normal_(0.0, 1.0, generator=gen)


class _Storage:
    """A transfer client whose storage is instantaneous: what is timed is this side of it."""

    def SaveKvCaches(self, uris, buffers):
        return client_types.ClientErrorCode.ER_OK, uris

    def LoadKvCaches(self, uris, buffers):
        return client_types.ClientErrorCode.ER_OK


def _prepare_blocks(case, seed):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    dtype, T, E, B = DTYPES[case["dtype"]], case["manager_block"], case["engine_block"], case["blocks"]
    L, kv, D = case["layers"], case["kv"], case["row"]
    per_block = T // E
    pool_blocks = B * per_block + B * per_block // 4 + 8
    pool = _fill(torch.empty((L, kv, pool_blocks, E, D), dtype=dtype, device=DEVICE), gen)
    mla = kv == 1
    layers = {"layers.%d" % i: pool[i, 0] if mla else pool[i] for i in range(L)}
    engine_blocks = np.random.default_rng(seed).permutation(pool_blocks)[:B * per_block].reshape(B, per_block)
    slots = (engine_blocks[:, :, None] * E + np.arange(E)).reshape(B, T)
    staging_order = np.random.default_rng(seed + 1).permutation(B)
    state = {"kind": case["kind"], "save": case["save"], "pool": pool, "T": T, "D": D}
    if E > 1:
        info = connector.register_kv_caches(layers, T, E, use_mla=mla)
        table = info.all_kvcache_ptr_tensor_gpu
    else:  # page size 1: one array of token rows per layer and K/V
        info = None
        table = torch.tensor([pool[i, j].data_ptr() for i in range(L) for j in range(kv)], dtype=torch.int64).to(DEVICE)
    if case["kind"] == "task":
        allocator = CopyBufferAllocator(DEVICE, dtype, [L, kv, T, D], B)
        if not case["save"]:
            _fill(allocator._raw_buffer, gen)
        state.update(
            staging=allocator._raw_buffer, ready=torch.cuda.Event(), index=slots.tolist(),
            manager=connector.DataTransferManager(info, T, allocator, _Storage()),
            uris=["file:///kv/%d?blkid=%d&size=%d" % (seed, b, _block_bytes(case)) for b in range(B)])
        return state
    staging = torch.empty((B, L, kv, T, D), dtype=dtype, device=DEVICE)
    if not case["save"]:
        _fill(staging, gen)
    state.update(staging=staging, table=table, form=case["index"], run=E)
    if case["index"] == "list":
        state.update(index=slots.reshape(-1).tolist(), order=staging_order.tolist())
    else:
        index = slots if case["index"] == "slots" else engine_blocks * E
        state.update(index=torch.from_numpy(index.astype(np.int32)).reshape(-1).to(DEVICE),
                     order=torch.from_numpy(staging_order.astype(np.int32)).to(DEVICE))
    return state


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("task", "copy"):
        return _prepare_blocks(case, seed)
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    if kind == "keys":
        dtype = torch.int64 if case["bits"] == 64 else torch.int32
        state = {"kind": kind, "block": case["block"], "offsets": None}
        if case["shortest"] == case["longest"]:
            shape = (case["requests"], case["longest"])
        else:
            offsets = _offsets(_lengths(case, seed))
            state["offsets"] = torch.from_numpy(offsets).to(DEVICE)
            shape = (int(offsets[-1]),)
        state["tokens"] = torch.randint(0, VOCAB, shape, dtype=dtype, device=DEVICE, generator=gen)
        return state
    if kind == "chain":
        offsets = _offsets(_lengths(case, seed))
        digests = torch.randint(-2**63, 2**63 - 1, (int(offsets[-1]),), dtype=torch.int64, device=DEVICE, generator=gen)
        return {"kind": kind, "digests": digests, "offsets": torch.from_numpy(offsets).to(DEVICE)}
    if kind == "sha":
        rng = random.Random(seed)
        n = case["characters"]
        return {"kind": kind, "strings": ["%0*x" % (n, rng.getrandbits(4 * n)) for _ in range(case["strings"])]}
    # select: requests share prefixes with 16 templates, and what the manager holds already is a prefix of each. Who shares
    # how much belongs to the case, so that every seed leaves as many blocks to save; the seed deals out keys and order.
    R, n = case["requests"], case["blocks"]
    rng = np.random.default_rng(R * n)
    which, shared = rng.integers(0, 16, size=R), (n * rng.random(R) ** 2).astype(np.int64)
    held_of_template = (n * case["saved"] * rng.random(16)).astype(np.int64)[which]
    held_of_request = (n * case["saved"] * rng.random(R)).astype(np.int64)
    held = np.where(held_of_template < shared, held_of_template, np.maximum(shared, held_of_request))
    rng = np.random.default_rng(seed)
    order = rng.permutation(R)
    keys = rng.integers(-2**63, 2**63 - 1, size=(R, n), dtype=np.int64)
    templates = rng.integers(-2**63, 2**63 - 1, size=(16, n), dtype=np.int64)
    keys = np.where(np.arange(n) < shared[:, None], templates[which], keys)[order]
    saved = (np.arange(n) < held[:, None])[order]
    return {"kind": kind, "keys": torch.from_numpy(keys.reshape(-1)).to(DEVICE),
            "saved": torch.from_numpy(saved.reshape(-1)).to(DEVICE)}


# ------------------------------------------------------------------------------------------------ one pass

def run(state):
    kind = state["kind"]
    if kind == "keys":
        return hashing.hash_tokens(state["tokens"], state["block"], token_offsets=state["offsets"])
    if kind == "chain":
        return hashing.apply_prefix_hash(state["digests"], state["offsets"])
    if kind == "sha":
        return hashing.sha256_to_int64(state["strings"], device=DEVICE)
    if kind == "select":
        indices, count = save_selection.select_save_indices(state["keys"], state["saved"])
        return indices[:int(count.item())]  # the caller sizes its transfer tasks by the count
    if kind == "task":
        manager, results = state["manager"], []
        done = connector.MultiResult(1, results.extend)
        if state["save"]:
            state["ready"].record()  # the forward pass that wrote the cache
            manager.save_task(done, 0, state["uris"], state["index"], state["ready"])
        else:
            manager.load_task(done, 0, state["uris"], state["index"])
        codes = np.array([int(code) for code in results[0]], dtype=np.int64)
        return {"blocks": state["staging"] if state["save"] else state["pool"], "codes": codes}
    operands = (state["table"], state["staging"], state["index"], state["order"], state["T"], state["D"])
    if state["form"] == "table":
        call = bgs.paged_gather_kv_caches if state["save"] else bgs.paged_scatter_kv_caches
        call(*operands, state["run"])
    else:
        call = bgs.batch_gather_kv_caches if state["save"] else bgs.batch_scatter_kv_caches
        call(*operands)
    return state["staging"] if state["save"] else state["pool"]


# ------------------------------------------------------------------------------------------------ bounds

def work(case):
    """Bytes: every input read once, every output written once. Operations: the steps of the recurrence (five whole-number
    operations each), the rounds of SHA-256; moving blocks has none."""
    kind = case["kind"]
    if kind == "keys":
        lengths = _lengths(case, 0)
        tokens, keys = int(lengths.sum()), int((lengths // case["block"]).sum())
        return {"bytes": tokens * case["bits"] // 8 + 8 * keys + 8 * (case["requests"] + 1), "flops": 5 * tokens}
    if kind == "chain":
        digests = int(_lengths(case, 0).sum())
        return {"bytes": 16 * digests + 8 * (case["requests"] + 1), "flops": 5 * digests}
    if kind == "sha":
        chunks = (case["characters"] + 8) // 64 + 1
        return {"bytes": case["strings"] * (case["characters"] + 16) + 8, "flops": case["strings"] * chunks * 64 * 30}
    if kind == "select":
        n = case["requests"] * case["blocks"]
        return {"bytes": n * (8 + 1) + int(n * (1 - case["saved"])) * 4 + 4, "flops": 0}
    entries = case["blocks"] * (1 + case["manager_block"] // (case["engine_block"] if case.get("index") == "table" else 1))
    return {"bytes": 2 * case["blocks"] * _block_bytes(case) + 4 * entries, "flops": 0}


def tolerance(case):
    return "exact"
