"""Block keys on the GPU: the manager's token hashing and its siblings, batched.

    hash_tokens / gen_key_vector   GenKeyVector        kv_cache_manager/manager/cache_manager.cc:76-87
                                   hashInt64Array      kv_cache_manager/manager/hash_util.h:14-24
    apply_prefix_hash              ApplyPrefixHash     kv_cache_manager/optimizer/trace_converter/trace_util.cc:47-56
    sha256_to_int64                _sha256_to_int64    kv_cache_manager/py_connector/sglang/connector.py:397-401
    prepare_block_keys             _prepare_block_keys kv_cache_manager/py_connector/sglang/connector.py:403-415

A connector that computes keys here can send `block_keys` instead of `token_ids`; the manager prefers them
(kv_cache_manager/manager/cache_manager.cc:306-318) and the keys are bit-identical to the ones it would compute.
"""
import threading
from array import array
from collections import deque
from itertools import accumulate
from typing import List, Optional, Sequence, Tuple

import torch

from . import _lib
from ._torch_util import lib, ptr, require_cuda, stream_handle

try:  # one C loop over a list of strings; absent only when the package was not built with its build.py
    from ._kvcm_pylist import pack_strings as _pack_strings, pack_strings_into as _pack_into, strings_size as _strings_size
except ImportError:  # host-side convenience only: the strings then go through Python
    _pack_strings = _pack_into = _strings_size = None


def _require_offsets(t, name, device, entries=None):
    """Offsets are read by the kernel as they are: int64, 1-D, on the tokens' device, R+1 entries."""
    require_cuda(t, name)
    n = t.numel()
    if t.dtype != torch.int64 or t.dim() != 1 or n < 1:
        raise ValueError(f"{name} must be a 1-D int64 tensor of R+1 entries")
    if t.device != device:
        raise ValueError(f"{name} is on {t.device}, the tokens on {device}")
    if entries is not None and n != entries:
        raise ValueError(f"{name} has {n} entries, expected {entries}")
    return n


def hash_tokens(tokens: torch.Tensor, block_size: int, token_offsets: Optional[torch.Tensor] = None,
                seed: int = 0, keys: Optional[torch.Tensor] = None,
                key_offsets: Optional[torch.Tensor] = None) -> Tuple[torch.Tensor, torch.Tensor]:
    """Parent-chained block keys of R requests in one launch.

    tokens: int64 or int32 device tensor, [R, L] (uniform lengths) or flat with token_offsets [R+1].
    Returns (keys, key_offsets): request r owns keys[key_offsets[r]:key_offsets[r+1]], len_r // block_size of
    them (a trailing partial block yields no key, cache_manager.cc:78). Offsets that reach beyond `tokens`, or keys beyond
    `keys`, are never followed: such a request is left out, and where the call waits for the number of keys it raises
    ValueError. Asynchronous on the current stream when
    `keys` and `key_offsets` are passed in (or the batch is a 2-D tensor); otherwise the call returns once the number of
    keys is known on the host, which does not wait for the keys themselves.
    """
    require_cuda(tokens, "tokens")
    if tokens.dtype not in (torch.int64, torch.int32):
        raise ValueError("tokens must be int64 or int32")
    if int(block_size) <= 0:
        raise ValueError("block_size must be positive")
    tokens = tokens.contiguous()
    block_size = int(block_size)
    if token_offsets is None:
        if tokens.dim() != 2:
            raise ValueError("tokens must be [R, L] when token_offsets is not given")
        R = tokens.shape[0]
        total = R * (tokens.shape[1] // block_size)
    else:
        R, total = _require_offsets(token_offsets, "token_offsets", tokens.device) - 1, None
        off = token_offsets.contiguous()
    if key_offsets is not None:
        _require_offsets(key_offsets, "key_offsets", tokens.device, R + 1)
        key_offsets = key_offsets.contiguous()
    if keys is not None:
        require_cuda(keys, "keys")
        if keys.dtype != torch.int64 or keys.device != tokens.device or not keys.is_contiguous():
            raise ValueError("keys must be a contiguous int64 tensor on the tokens' device")
        if total is not None and keys.numel() < total:
            raise ValueError(f"keys holds {keys.numel()} entries, the batch yields {total}")
    if token_offsets is None:  # equally long requests: one launch, which also writes the key offsets
        new_offsets = None
        if keys is None:
            keys = torch.empty(total, dtype=torch.int64, device=tokens.device)
        if total == 0:  # no request holds a full block: nothing to launch (GenKeyVector returns an empty vector)
            return keys, (torch.zeros(R + 1, dtype=torch.int64, device=tokens.device) if key_offsets is None
                          else key_offsets)
        if key_offsets is None:
            new_offsets = torch.empty(R + 1, dtype=torch.int64, device=tokens.device)
        rc = lib().kvcm_hip_hash_tokens_2d(ptr(tokens), tokens.element_size(), R, tokens.shape[1], block_size, int(seed),
                                           ptr(keys), ptr(key_offsets), ptr(new_offsets), stream_handle(tokens.device))
        _lib.check(rc, "kvcm_hip_hash_tokens_2d")
        return keys, (new_offsets if key_offsets is None else key_offsets)
    stream = stream_handle(tokens.device)
    if key_offsets is None and R == 0:
        key_offsets = torch.zeros(1, dtype=torch.int64, device=tokens.device)
    if keys is None and key_offsets is None:
        return _hash_and_count(tokens, off, R, block_size, seed, stream)
    if key_offsets is None:
        key_offsets = torch.empty(R + 1, dtype=torch.int64, device=tokens.device)
        _launch_offsets(tokens, off, R, block_size, keys.numel(), key_offsets, None, stream)
    if keys is None:
        total = int(key_offsets[-1].item())
        keys = torch.empty(total, dtype=torch.int64, device=tokens.device)
        if total == 0:
            return keys, key_offsets
    _launch_keys(tokens, off, R, block_size, seed, keys, key_offsets, stream)
    return keys, key_offsets


def _launch_offsets(tokens, off, R, block_size, n_keys, key_offsets, pending, stream):
    ws, ws_bytes = None, 0
    if R > 32768:  # fewer need no workspace
        ws_bytes = lib().kvcm_hip_key_offsets_workspace_bytes(R)
        ws = torch.empty(ws_bytes // 8, dtype=torch.int64, device=tokens.device)
    rc = lib().kvcm_hip_key_offsets_checked(off.data_ptr(), R, block_size, tokens.numel(), n_keys, ptr(ws), ws_bytes,
                                            key_offsets.data_ptr(), ptr(pending), stream)
    if rc:
        _lib.check(rc, "kvcm_hip_key_offsets_checked")


def _launch_keys(tokens, off, R, block_size, seed, keys, key_offsets, stream, pending=None):
    """With `pending` the launch writes key_offsets, and their last into that pinned word, itself."""
    if pending is not None:
        rc = lib().kvcm_hip_hash_tokens_counted(tokens.data_ptr(), tokens.element_size(), tokens.numel(), off.data_ptr(), R,
                                                block_size, int(seed), keys.data_ptr(), keys.numel(), key_offsets.data_ptr(),
                                                pending.data_ptr(), stream)
        if rc:
            _lib.check(rc, "kvcm_hip_hash_tokens_counted")
        return
    rc = lib().kvcm_hip_hash_tokens_checked(tokens.data_ptr(), tokens.element_size(), tokens.numel(), off.data_ptr(), R,
                                            block_size, int(seed), keys.data_ptr(), keys.numel(), key_offsets.data_ptr(), stream)
    if rc:
        _lib.check(rc, "kvcm_hip_hash_tokens_checked")


# Pinned words that a launched kernel has yet to write and nobody waits for any more. torch's pinned-memory pool knows
# nothing of that kernel, so a word is dropped only once its stream has run dry, and never if the stream cannot say so.
_owed = {}


def _settle(word, device):
    _owed[id(word)] = word
    try:
        torch.cuda.current_stream(device).synchronize()
    except Exception:
        return
    del _owed[id(word)]


# Keys up to which the buffer is allocated by what the token count bounds, before the number of keys is known: 256 MiB, a
# thousandth of the device's memory, which the call needs for itself even if the offsets name few of the tokens. Waiting for
# the number first costs 8 to 30 us: 2^22 keys of 16-token blocks 116 / 124 us, 2^23 218 / 227, 2^24 405 / 440.
_KEYS_AHEAD = 1 << 25


def _counted_by_the_hash(R, n_tokens):
    """Whether the hash launch makes the key offsets itself. That saves a launch, but the total comes later out of the larger
    kernel, the more so the more requests there are, and where a call waits longer for it than for the keys nothing is saved. us a
    call, two launches / one: 600 requests of 50 to 100 tokens 16.8 / 16.5, 1000: 16.5 / 16.9, 2500: 16.9 / 18.3; 1500 of 350 to 700
    17.1 / 17.2, of 450 to 900 18.1 / 17.4; 2500 of 350 to 700 17.9 / 18.3, of 450 to 900 18.5 / 18.1."""
    return R <= 640 or (R <= _lib.COUNT_KEYS_UP_TO and n_tokens >= 576 * R)


def _hash_and_count(tokens, off, R, block_size, seed, stream):
    """(keys, key_offsets) of R > 0 requests when the caller brings neither. The total is on its way to the host while the
    keys are being computed into a buffer of the size that the token count bounds: nobody waits for the hash kernel, and the
    hash kernel waits for nobody. The keys returned own their bytes, and at most one key per request more (as many trailing
    partial blocks as there are requests), however much of `tokens` the offsets leave out."""
    if stream and torch.cuda.is_current_stream_capturing():
        raise RuntimeError("hash_tokens with token_offsets waits for the number of keys, which a graph cannot: pass keys and "
                           "key_offsets to capture it")
    key_offsets = torch.empty(R + 1, dtype=torch.int64, device=tokens.device)
    most = tokens.numel() // block_size
    keys = torch.empty(most, dtype=torch.int64, device=tokens.device) if most <= _KEYS_AHEAD else None
    pending = torch.empty(1, dtype=torch.int64, pin_memory=True)
    try:
        if keys is not None and most and _counted_by_the_hash(R, tokens.numel()):
            _launch_keys(tokens, off, R, block_size, seed, keys, key_offsets, stream, pending)
        else:
            _launch_offsets(tokens, off, R, block_size, most, key_offsets, pending, stream)
            if keys is not None and most:
                _launch_keys(tokens, off, R, block_size, seed, keys, key_offsets, stream)
        rc = lib().kvcm_wait_value(pending.data_ptr(), stream)
        if rc:
            _lib.check(rc, "kvcm_wait_value")
    except BaseException:  # an interrupt as much as an error: the kernel may still be to come
        _settle(pending, tokens.device)
        raise
    total = pending.item()
    if not 0 <= total <= most:
        raise ValueError(f"token_offsets name blocks of {block_size} tokens beyond the {tokens.numel()} that tokens holds")
    if keys is None:
        keys = torch.empty(total, dtype=torch.int64, device=tokens.device)
        if total:
            _launch_keys(tokens, off, R, block_size, seed, keys, key_offsets, stream)
        return keys, key_offsets
    return keys[:total] if most - total <= R else keys[:total].clone(), key_offsets


def gen_key_vector(tokens, block_size: int, device=None) -> List[int]:
    """GenKeyVector for one request, with the reference's list-in / list-out shape."""
    if isinstance(tokens, torch.Tensor):
        t = tokens.reshape(1, -1)
        if not t.is_cuda:
            t = t.to(device or "cuda")
    else:
        t = torch.tensor(list(tokens), dtype=torch.int64, device=device or "cuda").reshape(1, -1)
    if t.shape[1] < block_size:
        return []
    keys, _ = hash_tokens(t, block_size)
    return keys.tolist()


def apply_prefix_hash(hash_ids: torch.Tensor, offsets: Optional[torch.Tensor] = None) -> torch.Tensor:
    """keys[i] = fold of hash_ids[0..i] per sequence (sequence r = hash_ids[offsets[r]:offsets[r+1]])."""
    require_cuda(hash_ids, "hash_ids")
    if hash_ids.dtype != torch.int64:
        raise ValueError("hash_ids must be int64")
    ids, device = hash_ids.contiguous(), hash_ids.device
    n, R = ids.numel(), 1
    if offsets is None:
        offsets = torch.tensor([0, n], dtype=torch.int64, device=device)
    else:
        R = _require_offsets(offsets, "offsets", device) - 1
        offsets = offsets.contiguous()
    keys = torch.empty(ids.shape, dtype=torch.int64, device=device)
    at = offsets.data_ptr()
    rc = lib().kvcm_hip_hash_tokens_checked(ids.data_ptr(), 8, n, at, R, 1, 0, keys.data_ptr(), n, at, stream_handle(device))
    if rc:
        _lib.check(rc, "kvcm_hip_hash_tokens_checked")
    return keys


# Bytes of packed strings up to which the kernel reads them where they are packed, in pinned host memory: a copy in front of it
# takes longer than the reads do, and from pageable memory the caller waits for it and for all work in front of it. us per call, in
# place / copied: one string of 64 characters 12.6 / 21.9, 1024: 18.0 / 36.9, 16 384: 89 / 173, of 200 (3.4 MB): 161 / 376.
_PINNED_MOST = 4 << 20
# Packed strings that launched kernels have yet to read, oldest first, with the event behind each. Calls that find as many as this
# under way, or with whose own there would be more bytes than this, copy instead: what finished calls leave here until the next one
# comes is no more than that either.
_LENT_MOST = 64
_LENT_BYTES_MOST = 16 << 20
_lent = deque()
_lent_lock = threading.Lock()
_spare_events = {}  # device -> events whose strings have been given back


def _settled_event(device, size=0):
    """An event for the next `size` bytes of packed strings, or None if too many are under way; gives back what has been read."""
    with _lent_lock:
        while _lent and _lent[0][1].query():
            was, event, _ = _lent.popleft()
            _spare_events.setdefault(was, []).append(event)
        if len(_lent) >= _LENT_MOST or size + sum(pinned.numel() for _, _, pinned in _lent) > _LENT_BYTES_MOST:
            return None
        spare = _spare_events.get(device)
        return spare.pop() if spare else torch.cuda.Event()


def _sha256_in_place(data, device):
    """The keys of a plain list or tuple of str or bytes, which the kernel reads in pinned memory; None if it has to be copied."""
    size = _strings_size(data)
    if size is None or size > _PINNED_MOST or torch.cuda.is_current_stream_capturing():
        return None
    pinned = torch.empty(size, dtype=torch.uint8, pin_memory=True)
    at = pinned.data_ptr()
    n = _pack_into(data, at, size)
    if n is None:  # the list changed in between
        return None
    out = torch.empty(n, dtype=torch.int64, device=device)
    require_cuda(out, "device")
    event = _settled_event(out.device, size)
    if event is None:
        return None
    stream = torch.cuda.current_stream(out.device)
    try:
        rc = lib().kvcm_hip_sha256_first8_be(at + 8 * (n + 1), at, n, out.data_ptr(), stream.cuda_stream)
        event.record(stream)
        with _lent_lock:
            _lent.append((out.device, event, pinned))
    except BaseException:  # an interrupt as much as an error: the kernel may still be to come
        _settle(pinned, out.device)
        raise
    _lib.check(rc, "kvcm_hip_sha256_first8_be")
    return out


def sha256_to_int64(data: Sequence[str], device="cuda") -> torch.Tensor:
    """int.from_bytes(sha256(s.encode('utf-8')).digest()[:8], 'big', signed=True) for every string, on the GPU."""
    packed = None
    if _pack_strings is not None and type(data) in (list, tuple) and data:
        out = _sha256_in_place(data, device)
        if out is not None:
            return out
        packed = _pack_strings(data)
    if packed is None:  # anything but a list of plain strings; a class of its own may iterate in its own way
        enc = [s.encode("utf-8") if isinstance(s, str) else bytes(s) for s in data]
        n = len(enc)
        if n == 0:
            return torch.empty(0, dtype=torch.int64, device=device)
        packed = bytearray(array("q", accumulate((len(e) for e in enc), initial=0)).tobytes() + b"".join(enc) + b"\0")
    else:
        n = len(data)
    d_packed = torch.frombuffer(packed, dtype=torch.uint8).to(device)  # offsets and bytes in one copy
    out = torch.empty(n, dtype=torch.int64, device=device)
    rc = lib().kvcm_hip_sha256_first8_be(ptr(d_packed) + 8 * (n + 1), ptr(d_packed), n, ptr(out), stream_handle(out.device))
    _lib.check(rc, "kvcm_hip_sha256_first8_be")
    return out


def prepare_block_keys(keys: List[str], prefix_keys: Optional[List[str]] = None,
                       device="cuda") -> Tuple[List[int], int, int]:
    """(int64 keys of prefix_keys + keys, len(prefix_keys), len(keys)) -- sglang/connector.py:403-415."""
    prefix_keys = list(prefix_keys) if prefix_keys is not None else []
    block_keys = sha256_to_int64(prefix_keys + list(keys), device=device).tolist()
    return block_keys, len(prefix_keys), len(keys)
