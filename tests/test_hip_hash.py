"""GPU parity: block keys from the HIP kernels, through the C-ABI, against the golden vectors and the CPU oracle.
Bit-exact int64."""
import hashlib

import numpy as np
import pytest
import torch

import _cases as cases
from _gpu import dev, host, sync

pytestmark = pytest.mark.gpu


def _h():
    from tair_kvcache_amd import hashing
    return hashing


def test_golden_c1(golden):
    tok = cases.tokens(4, 512, 151936, shared_rows=4, shared_len=256, seed=0)
    assert tok[0, :8].tolist() == golden["c1"]["tokens_row0_first8"]
    keys, off = _h().hash_tokens(dev(tok), 16)
    sync()
    assert host(off, np.int64).tolist() == [0, 32, 64, 96, 128]
    assert host(keys, np.int64).reshape(4, 32).tolist() == golden["c1"]["keys"]
    keys32, _ = _h().hash_tokens(dev(tok.astype(np.int32)), 16)
    sync()
    assert host(keys32, np.int64).reshape(4, 32).tolist() == golden["c1"]["keys"]


def test_golden_cases_single_requests(golden):
    for case in golden["cases"]:
        got = _h().gen_key_vector(case["tokens"], case["block_size"])
        assert got == case["keys"], case["name"]


def test_golden_prefix_chains(golden):
    for ch in golden["prefix_chains"]:
        if not ch["ids"]:
            continue
        got = _h().apply_prefix_hash(torch.tensor(ch["ids"], dtype=torch.int64, device="cuda"))
        sync()
        assert got.tolist() == ch["keys"]


@pytest.mark.parametrize("R,L,bs", [(64, 4096, 16), (1, 16, 16), (3, 1000, 16), (65, 256, 64), (130, 96, 8),
                                    (32, 1024, 128), (7, 333, 7), (5, 64, 1), (200, 40, 24)])
def test_uniform_batches_match_oracle(oracle, R, L, bs):
    print(f"hash case R={R} L={L} bs={bs}", flush=True)
    rng = np.random.default_rng(R * 1000 + L + bs)
    tok = rng.integers(-2**63, 2**63 - 1, size=(R, L), dtype=np.int64)  # full int64 range, both signs
    want, woff = oracle.hash_tokens(tok, bs)
    keys, off = _h().hash_tokens(dev(tok), bs)
    sync()
    assert (host(off, np.int64) == woff).all()
    assert (host(keys, np.int64) == want).all()


def test_ragged_batch_and_seed(oracle):
    rng = np.random.default_rng(3)
    lens = [0, 5, 16, 17, 160, 33, 1024, 31, 4096, 15, 48] + [int(x) for x in rng.integers(0, 700, size=120)]
    toks = [rng.integers(0, 152064, size=n, dtype=np.int64) for n in lens]
    flat = np.concatenate(toks)
    toff = np.zeros(len(lens) + 1, dtype=np.int64)
    np.cumsum(lens, out=toff[1:])
    for bs, seed in [(16, 0), (16, 12345), (5, -7), (64, 0)]:
        want, woff = oracle.hash_tokens(flat, bs, token_offsets=toff, seed=seed)
        keys, off = _h().hash_tokens(dev(flat), bs, token_offsets=dev(toff), seed=seed)
        sync()
        assert (host(off, np.int64) == woff).all()
        assert (host(keys, np.int64) == want).all(), (bs, seed)
    # int32 tokens, ragged (request starts at odd element offsets: 16-byte loads at 4-byte alignment)
    flat32 = flat.astype(np.int32)
    want, _ = oracle.hash_tokens(flat32, 16, token_offsets=toff)
    keys, _ = _h().hash_tokens(dev(flat32), 16, token_offsets=dev(toff))
    sync()
    assert (host(keys, np.int64) == want).all()


@pytest.mark.parametrize("dtype", [np.int64, np.int32])
def test_general_loader_path(oracle, force_general_hash_loader, dtype):
    """The loader form used when a workgroup's requests span 4 GiB or more (32-bit buffer offsets cannot reach),
    taken here from the test-only build in which every launch uses it, on a ragged batch whose last request ends exactly at the end of the buffer."""
    force_general_hash_loader(True)
    rng = np.random.default_rng(17)
    lens = [int(x) for x in rng.integers(0, 900, size=150)] + [64]
    flat = rng.integers(-2**31, 2**31 - 1, size=sum(lens), dtype=np.int64).astype(dtype)
    toff = np.zeros(len(lens) + 1, dtype=np.int64)
    np.cumsum(lens, out=toff[1:])
    want, woff = oracle.hash_tokens(flat, 16, token_offsets=toff)
    keys, off = _h().hash_tokens(dev(flat), 16, token_offsets=dev(toff))
    sync()
    assert (host(keys, np.int64) == want).all()


def test_config2_batch_prefix_property(oracle):
    """64 x 4096 tokens, half the requests share a 2048-token prefix: 128 leading keys shared, the rest distinct."""
    tok = cases.tokens(64, 4096, 128256, shared_rows=32, shared_len=2048, seed=0)
    keys, _ = _h().hash_tokens(dev(tok), 16)
    sync()
    k = host(keys, np.int64).reshape(64, 256)
    want, _ = oracle.hash_tokens(tok, 16)
    assert (k == want.reshape(64, 256)).all()
    assert (k[:32, :128] == k[0, :128]).all()
    assert len(np.unique(k[:, 128])) == 64 and len(np.unique(k[32:, 0])) == 32


@pytest.mark.parametrize("R,L,bs,vocab", [(32, 16384, 64, 152064), (128, 8192, 128, 129280)])
def test_config3_and_config4_batches(oracle, R, L, bs, vocab):
    tok = cases.tokens(R, L, vocab, shared_rows=R // 2, shared_len=(L * 3 // 4 // bs) * bs, seed=0)
    keys, _ = _h().hash_tokens(dev(tok), bs)
    sync()
    want, _ = oracle.hash_tokens(tok, bs, threads=8)
    assert (host(keys, np.int64) == want).all()


def test_config5_many_requests(oracle):
    tok = cases.tokens(1024, 1024, 152064, seed=0)
    keys, _ = _h().hash_tokens(dev(tok), 16)
    sync()
    want, _ = oracle.hash_tokens(tok, 16, threads=8)
    assert (host(keys, np.int64) == want).all()


def test_sha256_keys(oracle):
    rng = np.random.default_rng(6)
    strs = ["", "abc", "é-ü-漢字", "x" * 55, "y" * 56, "z" * 64, "w" * 119, "v" * 120, "u" * 1000]
    strs += ["%064x" % int(x) for x in rng.integers(0, 2**62, size=300)]
    got = _h().sha256_to_int64(strs).tolist()
    want = [int.from_bytes(hashlib.sha256(s.encode("utf-8")).digest()[:8], "big", signed=True) for s in strs]
    assert got == want
    assert got == oracle.sha256_first8_be(strs).tolist()
    keys, n_prefix, n_new = _h().prepare_block_keys(strs[10:20], prefix_keys=strs[:3])
    assert (n_prefix, n_new) == (3, 10) and keys == want[:3] + want[10:20]
    assert _h().prepare_block_keys([], None) == ([], 0, 0)


@pytest.mark.parametrize("helper", [True, False])
def test_sha256_of_every_kind_of_sequence(monkeypatch, helper):
    """Lists, tuples, generators; str, bytes and bytearray, also mixed; lengths around one and two 64-byte chunks, so that
    whole chunks start at every alignment; with the C packing loop and without."""
    if not helper:
        monkeypatch.setattr(_h(), "_pack_strings", None)
    strs = ["a" * k for k in list(range(0, 70)) + list(range(117, 131)) + [191, 192, 193, 700]]
    want = [int.from_bytes(hashlib.sha256(s.encode()).digest()[:8], "big", signed=True) for s in strs]
    forms = [strs, tuple(strs), (s for s in strs), [s.encode() for s in strs], [bytearray(s.encode()) for s in strs],
             [s if i % 2 else s.encode() for i, s in enumerate(strs)]]
    for form in forms:
        assert _h().sha256_to_int64(form).tolist() == want
    assert _h().sha256_to_int64([]).tolist() == [] and _h().sha256_to_int64(iter([])).tolist() == []
    with pytest.raises(UnicodeEncodeError):
        _h().sha256_to_int64(["\ud800"])


def test_sha256_of_a_list_that_iterates_in_its_own_way():
    class Backwards(list):
        def __iter__(self):
            return reversed(list.copy(self))

    strs = ["a", "bb", "", "\u00e9\u6f22\U0001f600" * 20]
    want = [int.from_bytes(hashlib.sha256(s.encode()).digest()[:8], "big", signed=True) for s in reversed(strs)]
    assert _h().sha256_to_int64(Backwards(strs)).tolist() == want
    assert _h().sha256_to_int64(strs).tolist() == want[::-1]


def test_bad_buffers_are_refused_on_the_host():
    """Short key buffers, offsets of the wrong type, length or device would be out-of-bounds device accesses: ValueError."""
    h = _h()
    tok = torch.zeros(4, 64, dtype=torch.int64, device="cuda")
    with pytest.raises(ValueError):
        h.hash_tokens(tok, 16, keys=torch.empty(15, dtype=torch.int64, device="cuda"))       # 16 keys needed
    with pytest.raises(ValueError):
        h.hash_tokens(tok, 16, keys=torch.empty(16, dtype=torch.int32, device="cuda"))
    with pytest.raises(ValueError):
        h.hash_tokens(tok, 16, keys=torch.empty(16, dtype=torch.int64))                      # keys on the host
    flat = tok.reshape(-1)
    off = torch.arange(5, dtype=torch.int64, device="cuda") * 64
    with pytest.raises(ValueError):
        h.hash_tokens(flat, 16, token_offsets=off.cpu())
    with pytest.raises(ValueError):
        h.hash_tokens(flat, 16, token_offsets=off.to(torch.int32))
    with pytest.raises(ValueError):
        h.hash_tokens(flat, 16, token_offsets=off, key_offsets=torch.zeros(4, dtype=torch.int64, device="cuda"))
    with pytest.raises(ValueError):
        h.apply_prefix_hash(flat, offsets=torch.tensor([0, 256], dtype=torch.int64))         # offsets on the host
    keys, _ = h.hash_tokens(flat, 16, token_offsets=off)                                     # and the good call works
    sync()
    assert keys.numel() == 16


@pytest.mark.parametrize("dtype", [np.int64, np.int32])
@pytest.mark.parametrize("shape", ["uniform", "uniform_odd_count", "ragged", "ragged_short", "two_lengths",
                                   "workgroup_on_every_cu", "every_cu_ragged", "every_cu_two_lengths",
                                   "short_and_long_workgroups"])
def test_many_requests_take_the_staged_key_path(oracle, dtype, shape):
    """In launches of thousands of requests the keys of 16-token blocks are collected in LDS and written out as rows of up to
    512 bytes by the loader waves: a sixteenth of a group per tile and the rest after the loop (8-byte tokens, 2048 to 8191
    requests; workgroups whose requests are shorter than 32 tiles store directly), or a whole group right after the barrier
    that closes it (8-byte tokens from 8192 requests, 4-byte tokens from 12 288, if they are long enough). Rows end where a
    request does; requests past a multiple of 64 are in a workgroup of their own. Every mixture against the oracle, exact."""
    rng = np.random.default_rng(5)
    lens = {
        "uniform": np.full(8192, 2048),                                # two whole groups per request
        "uniform_odd_count": np.full(8192 + 37, 1024 + 64 * 3 + 5),    # one group + three tiles + a tail; last workgroup partial
        "ragged": rng.integers(1100, 3000, size=8300),                 # first group whole for everyone, later ones not
        "ragged_short": rng.integers(0, 1500, size=9000),              # many workgroups with no whole group at all
        "two_lengths": np.where(np.arange(8192) % 64 < 32, 4096, 2048),  # half of every workgroup ends after two groups
        "workgroup_on_every_cu": np.full(16384 + 70, 1024 + 100),      # one group + a tile + a tail; last workgroup partial
        "every_cu_ragged": rng.integers(1100, 3000, size=16384 + 70),
        "every_cu_two_lengths": np.where(np.arange(16384) % 64 < 32, 3072, 1024),
        # workgroups of short requests (direct), of long ones (staged) and of both in one launch of the spread kernel
        "short_and_long_workgroups": np.where((np.arange(4096) // 64) % 3 == 0, 1536, np.where(np.arange(4096) % 5 == 0, 1024, 2560)),
    }[shape].astype(np.int64)
    toff = np.zeros(len(lens) + 1, dtype=np.int64)
    np.cumsum(lens, out=toff[1:])
    if dtype == np.int32:
        flat = rng.integers(-2**31, 2**31 - 1, size=int(toff[-1]), dtype=np.int64).astype(np.int32)
    else:
        flat = rng.integers(-2**63, 2**63 - 1, size=int(toff[-1]), dtype=np.int64)
    print(f"staged keys case {shape} {np.dtype(dtype).name}: {len(lens)} requests, {int(toff[-1])} tokens", flush=True)
    want, woff = oracle.hash_tokens(flat, 16, token_offsets=toff, seed=3, threads=8)
    keys = torch.full((len(want) + 64,), -7, dtype=torch.int64, device="cuda")    # room behind the keys: must stay untouched
    d_koff = dev(woff)
    got, off = _h().hash_tokens(dev(flat), 16, token_offsets=dev(toff), seed=3, keys=keys, key_offsets=d_koff)
    sync()
    assert (host(got, np.int64)[:len(want)] == want).all()
    assert (host(got, np.int64)[len(want):] == -7).all()


@pytest.mark.parametrize("dtype,R,bs", [(np.int64, 16384 + 70, 16), (np.int64, 8300, 16), (np.int32, 12288 + 70, 16),
                                         (np.int64, 300, 1), (np.int64, 2100, 8)])
def test_staged_keys_with_the_general_loader(oracle, force_general_hash_loader, dtype, R, bs):
    """The staged-key forms (spread and burst) are loader code as well: both with the loader that a workgroup spanning
    4 GiB of tokens would take, ragged requests, exact."""
    force_general_hash_loader(True)
    rng = np.random.default_rng(23)
    lens = rng.integers(1030, 2300, size=R).astype(np.int64)
    toff = np.zeros(R + 1, dtype=np.int64)
    np.cumsum(lens, out=toff[1:])
    flat = rng.integers(-2**31, 2**31 - 1, size=int(toff[-1]), dtype=np.int64).astype(dtype)
    print(f"staged keys, general loader: {R} requests of {np.dtype(dtype).name}, block size {bs}, {int(toff[-1])} tokens", flush=True)
    want, woff = oracle.hash_tokens(flat, bs, token_offsets=toff, threads=8)
    keys, off = _h().hash_tokens(dev(flat), bs, token_offsets=dev(toff))
    sync()
    assert (host(keys, np.int64) == want).all()



@pytest.mark.parametrize("dtype,R", [(np.int64, 2048 + 9), (np.int64, 10240 + 9), (np.int32, 12288 + 9), (np.int64, 2047)])
def test_key_offsets_with_gaps_and_odd_starts(oracle, dtype, R):
    """Keys go where key_offsets says, wherever that is: odd first positions (a request's 512-byte rows then start on
    8-byte boundaries only) and gaps between the requests' ranges, which must stay untouched -- on both sides of the
    request counts at which the way keys are written changes."""
    rng = np.random.default_rng(31)
    lens = rng.integers(2100, 2300, size=R).astype(np.int64)
    lens[::7] = 1024 + 48                                                # some requests end early in every workgroup
    toff = np.zeros(R + 1, dtype=np.int64)
    np.cumsum(lens, out=toff[1:])
    flat = rng.integers(-2**31, 2**31 - 1, size=int(toff[-1]), dtype=np.int64).astype(dtype)
    want, woff = oracle.hash_tokens(flat, 16, token_offsets=toff, seed=-5, threads=8)
    counts = lens // 16
    gaps = rng.integers(0, 4, size=R)
    koff = np.zeros(R + 1, dtype=np.int64)
    koff[0] = 1
    koff[1:] = 1 + np.cumsum(counts + gaps)
    print(f"gapped key offsets: {R} requests of {np.dtype(dtype).name}, {int(koff[-1])} key slots", flush=True)
    keys = torch.full((int(koff[-1]) + 64,), -7, dtype=torch.int64, device="cuda")
    got, _ = _h().hash_tokens(dev(flat), 16, token_offsets=dev(toff), seed=-5, keys=keys, key_offsets=dev(koff))
    sync()
    got = host(got, np.int64)
    expect = np.full(got.shape, -7, dtype=np.int64)
    for r in range(R):
        expect[koff[r]:koff[r] + counts[r]] = want[woff[r]:woff[r + 1]]
    assert (got == expect).all()


@pytest.mark.parametrize("bs,dtype", [(1, np.int64), (8, np.int64), (32, np.int64), (64, np.int64), (8, np.int32),
                                      (1, np.int32), (128, np.int64)])
def test_staged_keys_at_other_block_sizes(oracle, bs, dtype):
    """In launches of many requests the keys of 1-, 8-, 32-, 64- and 128-token blocks are staged too (a group is as many
    tiles as yield 64 keys per request: 1, 8, 32, 64, 128 tiles) and leave a group at a time. Ragged requests of one to three
    groups, some ending early, the last workgroup partial; exact against the oracle, spare key slots untouched."""
    group_tokens = 64 * max(bs, 1) if bs > 1 else 64
    rng = np.random.default_rng(41 + bs)
    R = (10240 if dtype == np.int64 else 12288) + 37   # past every threshold of the launch rule
    lens = rng.integers(group_tokens + 70, (3 if bs < 128 else 1.5) * group_tokens, size=R).astype(np.int64)
    lens[::9] = group_tokens // 2 + 5
    toff = np.zeros(R + 1, dtype=np.int64)
    np.cumsum(lens, out=toff[1:])
    flat = rng.integers(-2**31, 2**31 - 1, size=int(toff[-1]), dtype=np.int64).astype(dtype)
    print(f"staged keys, block size {bs}: {R} requests of {np.dtype(dtype).name}, {int(toff[-1])} tokens", flush=True)
    want, woff = oracle.hash_tokens(flat, bs, token_offsets=toff, seed=11, threads=8)
    keys = torch.full((len(want) + 64,), -7, dtype=torch.int64, device="cuda")
    got, off = _h().hash_tokens(dev(flat), bs, token_offsets=dev(toff), seed=11, keys=keys, key_offsets=dev(woff))
    sync()
    got = host(got, np.int64)
    assert (got[:len(want)] == want).all()
    assert (got[len(want):] == -7).all()


@pytest.mark.parametrize("dtype,R,bs", [(np.int64, 31, 1), (np.int64, 32, 1), (np.int64, 100, 1), (np.int32, 63, 1),
                                        (np.int32, 64, 1), (np.int64, 2048, 16), (np.int64, 8192, 16), (np.int64, 4096, 128),
                                        (np.int64, 2048, 8), (np.int64, 64, 16), (np.int64, 64, 32), (np.int64, 64, 64)])
def test_requests_that_end_inside_a_group_of_staged_keys(oracle, dtype, R, bs):
    """Staged keys leave as rows of pairs: requests with an odd number of keys, with none, with one key into a new group and
    with one key less than a group, beside requests that go on, so that every kind of row end meets every step of the
    drain; and on both sides of the request counts at which keys are staged. Spare key slots stay untouched."""
    rng = np.random.default_rng(1000 * bs + R)
    ends = np.array([0, 1, 2, 3, 31, 32, 33, 62, 63, 64, 65, 66, 127, 128, 129, 131])    # in keys
    nkeys = ends[rng.integers(0, len(ends), size=R)]
    nkeys[::64] = 131                                          # a long one in every workgroup
    if R > 2000:
        nkeys[64:128] = rng.integers(0, 20, size=64)           # one workgroup of short requests only
    lens = nkeys * bs + rng.integers(0, bs, size=R)
    toff = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    flat = rng.integers(-2**31, 2**31, size=max(int(toff[-1]), 1), dtype=np.int64).astype(dtype)
    want, woff = oracle.hash_tokens(flat, bs, token_offsets=toff, seed=5, threads=8)
    keys = torch.full((len(want) + 64,), -7, dtype=torch.int64, device="cuda")
    got, _ = _h().hash_tokens(dev(flat), bs, token_offsets=dev(toff), seed=5, keys=keys, key_offsets=dev(woff))
    sync()
    got = host(got, np.int64)
    assert (got[:len(want)] == want).all()
    assert (got[len(want):] == -7).all()


@pytest.mark.parametrize("general_loader", [False, True])
@pytest.mark.parametrize("bs", [8, 16, 32, 64, 128])
def test_raw_tiles_of_4_byte_tokens(oracle, force_general_hash_loader, bs, general_loader):
    """Launches of 12 288 requests or more of 4-byte tokens use tiles of 128 RAW tokens per request (the chain wave
    sign-extends and adds the constant itself) and write their keys as whole rows. Request lengths sit on and around
    the tile width (64, 127, 128, 129, 192, 256, ...), on multiples of a key group, and in between; every workgroup
    mixes them; tokens cover the whole signed 32-bit range. Both loaders. Exact against the oracle."""
    force_general_hash_loader(general_loader)
    rng = np.random.default_rng(41 + bs)
    R = 12288 + 77                                   # the last workgroup is partial
    group = 64 * bs                                  # tokens that yield one group of staged keys
    menu = np.array([0, 1, bs - 1, bs, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 257, 384, 511, 512,
                     group - 1, group, group + 1, group + 128, group + 129, 2 * group, 2 * group + 64 + bs])
    lens = menu[rng.integers(0, len(menu), size=R)].astype(np.int64)
    lens[rng.random(R) < 0.3] = rng.integers(0, 2 * group + 300)      # and anything in between
    lens[:64] = 2 * group + 128                      # one workgroup of equal, whole requests: every group staged
    lens[64:128] = np.where(np.arange(64) % 2 == 0, group + 128, 2 * group)
    scale = max(1, int(lens.sum() // 40_000_000) + 1)                 # keep the launch under ~160 MB of tokens
    if scale > 1:
        lens[128:] = lens[128:] // scale
    toff = np.zeros(R + 1, dtype=np.int64)
    np.cumsum(lens, out=toff[1:])
    flat = rng.integers(-2**31, 2**31, size=int(toff[-1]), dtype=np.int64).astype(np.int32)
    flat[:16] = [-2**31, 2**31 - 1, -1, 0, 1, -2, 2**31 - 2, -2**31 + 1] * 2
    print(f"raw tiles: bs={bs} general_loader={general_loader} R={R} tokens={int(toff[-1])}", flush=True)
    want, woff = oracle.hash_tokens(flat, bs, token_offsets=toff, seed=-3)
    keys = torch.full((len(want) + 64,), -7, dtype=torch.int64, device="cuda")
    got, off = _h().hash_tokens(dev(flat), bs, token_offsets=dev(toff), seed=-3, keys=keys, key_offsets=dev(woff))
    sync()
    got = host(got, np.int64)
    assert (got[:len(want)] == want).all()
    assert (got[len(want):] == -7).all()
    # the mean length decides above; through the entry that does not know it, requests count as long and tiles are raw
    keys.fill_(-7)
    d_flat, d_toff, d_koff = dev(flat), dev(toff), dev(woff)
    rc = _h().lib().kvcm_hip_hash_tokens_i32(d_flat.data_ptr(), d_toff.data_ptr(), R, bs, -3, keys.data_ptr(), d_koff.data_ptr(),
                                             torch.cuda.current_stream().cuda_stream)
    sync()
    got = host(keys, np.int64)
    assert rc == 0 and (got[:len(want)] == want).all() and (got[len(want):] == -7).all()


@pytest.mark.parametrize("R,L,bs", [(1, 16, 16), (63, 17, 16), (64, 130, 64), (65, 47, 24), (128, 128, 128), (129, 10, 3)])
def test_equally_long_requests_need_no_offset_arrays(oracle, R, L, bs):
    """[R, L] tokens in one launch: lengths with and without a trailing partial block, request counts around a workgroup's
    64, both token widths, key offsets written by the launch or given by the caller (with gaps between the requests)."""
    rng = np.random.default_rng(R * 131 + L)
    tok = rng.integers(-2**31, 2**31 - 1, size=(R, L), dtype=np.int64)
    want, woff = oracle.hash_tokens(tok, bs, seed=9)
    per = L // bs
    gaps = np.arange(R + 1, dtype=np.int64) * (per + 1)
    for dtype in (np.int64, np.int32):
        keys, off = _h().hash_tokens(dev(tok.astype(dtype)), bs, seed=9)
        spread = torch.full((R * (per + 1),), -7, dtype=torch.int64, device="cuda")
        _, same = _h().hash_tokens(dev(tok.astype(dtype)), bs, seed=9, keys=spread, key_offsets=dev(gaps))
        sync()
        assert (host(keys, np.int64) == want).all() and (host(off, np.int64) == woff).all()
        assert (host(same, np.int64) == gaps).all()
        got = host(spread, np.int64).reshape(R, per + 1)
        assert (got[:, :per] == want.reshape(R, per)).all() and (got[:, per] == -7).all()


@pytest.mark.parametrize("R", [1, 8, 9, 513, 8192, 8193, 32768, 32769])
def test_key_offsets_of_ragged_batches(oracle, R):
    """Offsets and keys when the caller passes neither, at the edges of the prefix-sum kernel (eight requests per thread,
    8192 per workgroup) and beyond the request count it is used for; some requests empty or shorter than a block."""
    rng = np.random.default_rng(R)
    lens = rng.integers(0, 70, size=R)
    toff = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    flat = rng.integers(0, 152064, size=max(int(toff[-1]), 1), dtype=np.int64)
    want, woff = oracle.hash_tokens(flat, 16, token_offsets=toff, threads=8)
    keys, off = _h().hash_tokens(dev(flat), 16, token_offsets=dev(toff))
    sync()
    assert (host(off, np.int64) == woff).all() and (host(keys, np.int64) == want).all()


def test_offsets_beyond_the_tokens_are_refused():
    """Offsets that name more blocks than the tokens can hold: nothing is written past the keys, and the call says so.
    (The tokens are the front of a larger array, so what the launch reads is its own.)"""
    flat = torch.zeros(4096, dtype=torch.int64, device="cuda")
    off = torch.arange(0, 4097, 512, dtype=torch.int64, device="cuda")
    with pytest.raises(ValueError):
        _h().hash_tokens(flat[:1024], 16, token_offsets=off)
    sync()


@pytest.mark.parametrize("general_loader", [False, True])
@pytest.mark.parametrize("dtype", [np.int64, np.int32])
@pytest.mark.parametrize("R", [17, 40001])   # the last request is whole blocks up to the end of the tokens
def test_offsets_are_not_followed_beyond_the_tokens(oracle, force_general_hash_loader, general_loader, dtype, R):
    """Offsets that reach beyond `tokens` although the number of blocks would fit, because most requests are shorter than a
    block: ValueError, as one launch counts the blocks and as two do. An overrun inside a trailing partial block costs no
    key and changes none. (All arrays are the front of larger ones, whose rest must not matter and must not change.)"""
    force_general_hash_loader(general_loader)
    rng = np.random.default_rng(R)
    n = 16 * R
    big = rng.integers(-2**31, 2**31, size=2 * n + 4096, dtype=np.int64).astype(dtype)
    tok = dev(big)[:n]
    toff = np.minimum(np.arange(R + 1) * 15, n).astype(np.int64)                 # no request holds a block ...
    for last, ok in ((n, True), (n + 3, True), (n + 16, False), (n + 2000, False)):
        toff[-1] = last                                                          # ... but the last one
        d_off = dev(toff)
        if not ok:
            with pytest.raises(ValueError):
                _h().hash_tokens(tok, 16, token_offsets=d_off)
            continue
        keys, off = _h().hash_tokens(tok, 16, token_offsets=d_off)
        sync()
        want, woff = oracle.hash_tokens(big, 16, token_offsets=toff, threads=8)
        assert (host(keys, np.int64) == want).all() and (host(off, np.int64) == woff).all(), last
    # what is asked to go into the caller's own buffer is left out, and marked where the offsets are this call's
    toff[-1] = n + 16
    room = torch.full((2 * R + 64,), -7, dtype=torch.int64, device="cuda")
    _, off = _h().hash_tokens(tok, 16, token_offsets=dev(toff), keys=room[:R])
    _h().hash_tokens(tok, 16, token_offsets=dev(toff), keys=room[:R], key_offsets=dev(np.zeros(R + 1, dtype=np.int64)))
    sync()
    assert (host(room, np.int64) == -7).all() and host(off, np.int64)[R - 1] == -1


@pytest.mark.parametrize("one_launch", [True, False])
@pytest.mark.parametrize("dtype,bs", [(np.int64, 16), (np.int32, 1), (np.int32, 7), (np.int64, 7)])
@pytest.mark.parametrize("R", [1, 16, 17, 271, 272, 273, 529, 1040, 1041, 1552, 1553, 4096, 4097])
def test_one_launch_counts_and_hashes(oracle, monkeypatch, one_launch, dtype, bs, R):
    """Ragged batches whose offsets the launch itself makes, at the edges of its workgroups (16 requests), of the offsets that a
    wave adds up at a time (256, and 1024 while more than 512 are left) and of the most it takes: keys, offsets, and requests that
    are not all there, any one of which, in front of a workgroup or its own, is found. The same as two launches."""
    monkeypatch.setattr(_h(), "_counted_by_the_hash", lambda R, n: one_launch and R <= 4096)
    rng = np.random.default_rng(R * bs)
    lens = rng.integers(0, 100, size=R)
    lens[R // 2] += 3 * bs
    toff = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    flat = rng.integers(-2**31, 2**31, size=int(toff[-1]) + 40, dtype=np.int64).astype(dtype)
    want, woff = oracle.hash_tokens(flat, bs, token_offsets=toff, threads=8)
    keys, off = _h().hash_tokens(dev(flat), bs, token_offsets=dev(toff))
    sync()
    assert (host(off, np.int64) == woff).all() and (host(keys, np.int64) == want).all()
    for r in {0, R // 2, R - 1}:
        far = toff.copy()
        far[r + 1] = len(flat) + bs                          # and whoever comes next begins there
        with pytest.raises(ValueError):
            _h().hash_tokens(dev(flat), bs, token_offsets=dev(far))
    sync()


@pytest.mark.parametrize("one_launch", [True, False])
@pytest.mark.parametrize("dtype", [np.int64, np.int32])
@pytest.mark.parametrize("bs,bad", [(1, 1), (1, 2), (1, 3), (16, 1), (16, 16), (16, 32), (16, 300), (7, 30)])
def test_offsets_whose_counts_add_up_to_more_than_63_bits(oracle, monkeypatch, one_launch, dtype, bs, bad):
    """Requests that name tokens far beyond the array, many enough that their counts would wrap to below zero and back, in front of
    sound ones, in the same workgroup and in later ones: nothing is written but the keys of requests that are all there and fit, at
    the exact place; everybody else gets the offset -1. (The key buffer is the middle of a larger one that must not change.)"""
    h = _h()
    rng = np.random.default_rng(bs + bad)
    n = 4096
    far = 2**62 + 2**40
    toff = [0, 16, 16 + 3 * bs, 0] + [far, 0] * bad + [5, 5 + 2 * bs, 300, 300 + bs, n] + [n] * 20 + [n - bs, n]
    R = len(toff) - 1
    flat = rng.integers(-2**31, 2**31, size=n, dtype=np.int64).astype(dtype)
    tok, off = dev(flat), dev(np.array(toff, dtype=np.int64))
    room = torch.full((3 * n,), -7, dtype=torch.int64, device="cuda")
    koff = torch.full((R + 1,), -9, dtype=torch.int64, device="cuda")
    word = torch.empty(1, dtype=torch.int64, pin_memory=True)
    stream = torch.cuda.current_stream().cuda_stream
    sync()
    if one_launch:
        h._launch_keys(tok, off, R, bs, 3, room[n:2 * n], koff, stream, word)
    else:
        h._launch_offsets(tok, off, R, bs, n, koff, word, stream)
        h._launch_keys(tok, off, R, bs, 3, room[n:2 * n], koff, stream)
    sync()
    want_room, want_koff, at, left_out = np.full(3 * n, -7, dtype=np.int64), [], 0, 0
    for a, b in zip(toff[:-1], toff[1:]):
        length = (b - a + 2**63) % 2**64 - 2**63                    # distances are formed in 64 bits
        count = max(0, length) // bs
        whole = count == 0 or (0 <= a and a + count * bs <= n)
        left_out += not whole
        fits = whole and at + count <= n
        want_koff.append(at if fits else -1)
        if fits and count:
            want_room[n + at:n + at + count], _ = oracle.hash_tokens(flat[a:a + count * bs].astype(np.int64)[None], bs, seed=3)
        at += count
    want_koff.append(min(at, 2**41))
    assert left_out and word.item() == -1
    assert host(koff, np.int64).tolist() == want_koff
    assert (host(room, np.int64) == want_room).all()
    monkeypatch.setattr(h, "_counted_by_the_hash", lambda R, n: one_launch)
    with pytest.raises(ValueError):
        h.hash_tokens(tok, bs, token_offsets=off)
    sync()


@pytest.mark.parametrize("general_loader", [False, True])
@pytest.mark.parametrize("dtype,bs", [(np.int64, 16), (np.int32, 7), (np.int64, 1), (np.int32, 16)])
@pytest.mark.parametrize("R", [20, 1000, 4200])
def test_offsets_that_go_back(oracle, force_general_hash_loader, general_loader, dtype, bs, R):
    """Token offsets that do not ascend: a request that ends in front of its start has no keys, and the ones behind it, wherever
    they begin (in front of their workgroup's first offset, behind its last), those of their own tokens."""
    force_general_hash_loader(general_loader)
    rng = np.random.default_rng(R * bs)
    n = 20000
    flat = rng.integers(-2**31, 2**31, size=n, dtype=np.int64).astype(dtype)
    toff = [n - 300]
    for r in range(R):
        toff.append(toff[-1] + int(rng.integers(0, 300)))
        if toff[-1] > n or rng.random() < 0.2:
            toff[-1] = int(rng.integers(0, max(1, min(n - 600, toff[-2]))))
    counts = [max(0, b - a) // bs for a, b in zip(toff[:-1], toff[1:])]
    koff = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    assert any(b < a for a, b in zip(toff[:-1], toff[1:])) and max(toff) <= n
    want = [oracle.hash_tokens(flat[None, a:a + c * bs].astype(np.int64), bs, seed=9)[0] for a, c in zip(toff, counts) if c]
    want = np.concatenate(want)
    tok, off = dev(flat), dev(np.array(toff, dtype=np.int64))
    keys = torch.full((len(want) + 64,), -7, dtype=torch.int64, device="cuda")
    _h().hash_tokens(tok, bs, token_offsets=off, seed=9, keys=keys, key_offsets=dev(koff))
    sync()
    assert (host(keys, np.int64)[:len(want)] == want).all() and (host(keys, np.int64)[len(want):] == -7).all()
    if koff[-1] <= n // bs:                                      # counted by the call as well
        got, goff = _h().hash_tokens(tok, bs, token_offsets=off, seed=9)
        sync()
        assert (host(got, np.int64) == want).all() and (host(goff, np.int64) == koff).all()


@pytest.mark.parametrize("general_loader", [False, True])
def test_keys_beyond_the_callers_buffer_are_left_out(oracle, force_general_hash_loader, general_loader):
    """A key buffer that holds the keys of some requests only: those are written, the slots behind the buffer are not; the
    same for a chain whose offsets name more digests than there are."""
    force_general_hash_loader(general_loader)
    rng = np.random.default_rng(3)
    lens = np.array([33, 0, 160, 15, 64, 700, 16])
    toff = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    flat = rng.integers(0, 152064, size=int(toff[-1]), dtype=np.int64)
    want, woff = oracle.hash_tokens(flat, 16, token_offsets=toff)
    for short in (1, 2, 44, 45, 46):
        room = torch.full((len(want) + 64,), -7, dtype=torch.int64, device="cuda")
        for koff in (None, dev(woff)):
            room.fill_(-7)
            _h().hash_tokens(dev(flat), 16, token_offsets=dev(toff), keys=room[:len(want) - short], key_offsets=koff)
            sync()
            got = host(room, np.int64)
            for r in range(len(lens)):
                fits = woff[r + 1] <= len(want) - short
                assert (got[woff[r]:woff[r + 1]] == (want[woff[r]:woff[r + 1]] if fits else -7)).all(), (short, r)
            assert (got[len(want):] == -7).all()
    chain, _ = oracle.hash_tokens(flat, 1, token_offsets=toff)
    got = _h().apply_prefix_hash(dev(flat)[:300], dev(toff))                     # requests 5 and 6 end beyond digest 300
    sync()
    assert got.shape == (300,) and (host(got, np.int64)[:272] == chain[:272]).all()


@pytest.mark.parametrize("fails", ["kvcm_hip_hash_tokens_checked", "kvcm_hip_hash_tokens_counted", "kvcm_wait_value"])
def test_the_word_a_kernel_has_yet_to_write_outlives_an_error(monkeypatch, fails):
    """A call that ends with an error, or is interrupted, between the launch that writes the number of keys into pinned memory
    and the wait for it: the stream has run dry before that memory can go to anybody else. (In front of a failing launch that
    takes its offsets there is the one that makes them; a launch that counts for itself is the first of its call.)"""
    from tair_kvcache_amd import _lib, _torch_util
    h = _h()

    class Failing:
        def __getattr__(self, name):
            if name != fails:
                return getattr(_torch_util.lib(), name)

            def entry(*args):
                if name == "kvcm_wait_value":
                    raise KeyboardInterrupt
                return _lib.ERR_INVALID_ARG
            return entry

    off = torch.arange(0, 8193, 64, dtype=torch.int64, device="cuda")
    tok = torch.zeros(8192, dtype=torch.int64, device="cuda")
    queued = torch.empty(1 << 28, dtype=torch.int8, device="cuda")
    monkeypatch.setattr(h, "lib", Failing)
    monkeypatch.setattr(h, "_counted_by_the_hash", lambda R, n: fails != "kvcm_hip_hash_tokens_checked")
    sync()
    for _ in range(64):                                       # some milliseconds of work in front of the kernel
        queued.zero_()
    with pytest.raises((_lib.KvcmError, KeyboardInterrupt)):
        h.hash_tokens(tok, 16, token_offsets=off)
    assert torch.cuda.current_stream().query() and not h._owed


@pytest.mark.parametrize("spare,bs", [(0, 16), (15, 16), (100_000, 16), (100_000, 1), (1 << 24, 1), ((1 << 25) + 64, 1)])
def test_keys_own_no_more_than_their_bytes(oracle, spare, bs):
    """The key buffer does not grow with tokens that the offsets leave out, be they fewer or more than what is allocated for
    before the number of keys is known."""
    rng = np.random.default_rng(spare)
    lens = rng.integers(0, 200, size=64)
    toff = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    flat = rng.integers(0, 152064, size=int(toff[-1]), dtype=np.int64)
    want, woff = oracle.hash_tokens(flat, bs, token_offsets=toff)
    tok = torch.zeros(len(flat) + spare, dtype=torch.int64, device="cuda")
    tok[:len(flat)] = dev(flat)
    torch.cuda.synchronize()
    keys, off = _h().hash_tokens(tok, bs, token_offsets=dev(toff))
    sync()
    assert (host(keys, np.int64) == want).all() and (host(off, np.int64) == woff).all()
    assert keys.untyped_storage().nbytes() <= 8 * (len(want) + len(lens))
    none, _ = _h().hash_tokens(tok, bs, token_offsets=torch.zeros(3, dtype=torch.int64, device="cuda"))
    assert none.numel() == 0 and none.untyped_storage().nbytes() <= 16


def test_a_call_that_waits_is_refused_under_capture_before_it_launches_anything(oracle):
    """Ragged offsets and no key buffer: the call would wait for a number that no graph delivers. It says so without spoiling
    the capture; with keys and offsets of the caller's it is captured, and every replay hashes the tokens of the day."""
    from tair_kvcache_amd import _lib
    rng = np.random.default_rng(8)
    lens = rng.integers(0, 300, size=70)
    toff = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    tok, off = torch.zeros(int(toff[-1]), dtype=torch.int64, device="cuda"), dev(toff)
    keys = torch.empty(len(tok) // 16, dtype=torch.int64, device="cuda")
    word = torch.full((1,), 5, dtype=torch.int64, pin_memory=True)
    _h().hash_tokens(tok, 16, token_offsets=off)
    sync()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        with pytest.raises(RuntimeError, match="key_offsets"):
            _h().hash_tokens(tok, 16, token_offsets=off)
        stream = torch.cuda.current_stream().cuda_stream
        rc = _lib.lib().kvcm_hip_key_offsets(off.data_ptr(), 70, 16, 1 << 40, keys.data_ptr(), word.data_ptr(), stream)
        assert rc > 0 and word.item() == 5
        word.fill_(-2**62)                                       # KVCM_PENDING
        assert _lib.lib().kvcm_wait_value(word.data_ptr(), stream) > 0
        _, koff = _h().hash_tokens(tok, 16, token_offsets=off, keys=keys)
    for _ in range(3):
        flat = rng.integers(0, 152064, size=len(tok), dtype=np.int64)
        tok.copy_(dev(flat))
        graph.replay()
        sync()
        want, woff = oracle.hash_tokens(flat, 16, token_offsets=toff)
        assert (host(koff, np.int64) == woff).all() and (host(keys, np.int64)[:len(want)] == want).all()


@pytest.mark.parametrize("dtype,bs,R,mean", [
    (np.int64, 8, 2048, 320), (np.int64, 16, 8192, 320), (np.int64, 32, 8192, 560), (np.int64, 64, 8192, 896),
    (np.int64, 128, 4096, 960), (np.int32, 8, 12288, 640), (np.int32, 16, 12288, 1024), (np.int32, 32, 12288, 1600),
    (np.int32, 64, 12288, 2304), (np.int32, 128, 12288, 2560), (np.int32, 1, 64, 129), (np.int32, 1, 2049, 129)])
def test_mean_lengths_on_both_sides_of_the_staging_rule(oracle, dtype, bs, R, mean):
    """Thousands of requests are staged from a mean length on: one token less, and exactly that many, from requests that are
    empty, shorter than a block, around a tile and several tiles long, in whatever workgroup. Spare key slots stay untouched."""
    rng = np.random.default_rng(bs + R)
    R += 9                                                     # the last workgroup is partial
    for n_tokens in (mean * R - 1, mean * R):
        menu = np.array([0, 1, bs - 1, bs, 63, 64, 65, 127, 128, 129, mean, 2 * mean, 3 * mean + 5])
        lens = menu[rng.integers(0, len(menu), size=R)].astype(np.int64)
        lens[:64] = 0                                          # a workgroup without a block
        short = n_tokens - int(lens.sum())                     # brought to the wanted sum a little at a time
        step = np.sign(short) * rng.integers(0, 2 * mean, size=R)
        step[:64] = 0
        done = np.cumsum(np.abs(np.maximum(step, -lens)))
        lens += np.where(done <= abs(short), np.maximum(step, -lens), 0)
        lens[-1] += max(0, n_tokens - int(lens.sum()))
        lens[np.argmax(lens)] += n_tokens - int(lens.sum())
        assert lens.sum() == n_tokens and lens.min() >= 0
        toff = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
        flat = rng.integers(-2**31, 2**31, size=n_tokens, dtype=np.int64).astype(dtype)
        want, woff = oracle.hash_tokens(flat, bs, token_offsets=toff, seed=7, threads=8)
        print(f"staging rule: bs={bs} {np.dtype(dtype).name} {R} requests, {n_tokens} tokens", flush=True)
        keys = torch.full((len(want) + 64,), -7, dtype=torch.int64, device="cuda")
        _h().hash_tokens(dev(flat), bs, token_offsets=dev(toff), seed=7, keys=keys, key_offsets=dev(woff))
        sync()
        got = host(keys, np.int64)
        assert (got[:len(want)] == want).all() and (got[len(want):] == -7).all()


@pytest.mark.parametrize("dtype", [np.int64, np.int32])
@pytest.mark.parametrize("R", [1, 2, 31, 32, 33, 63, 64, 65, 1024, 1025])
def test_block_size_1_equally_long_and_ragged(oracle, dtype, R):
    """A key per token: few or short equally long requests are stored by the chain wave itself, others staged; around 32
    requests of a workgroup, 16 workgroups and 8 tiles, with lengths that end inside a tile."""
    rng = np.random.default_rng(R)
    for length in (1, 63, 64, 65, 448, 511, 512, 513, 576, 600):
        for spread in (0, 1, 70, length):
            lens = np.maximum(0, length - rng.integers(0, spread + 1, size=R)).astype(np.int64)
            toff = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
            flat = rng.integers(-2**31, 2**31, size=max(int(toff[-1]), 1), dtype=np.int64).astype(dtype)
            want, woff = oracle.hash_tokens(flat, 1, token_offsets=toff, seed=7, threads=8)
            keys = torch.full((len(want) + 64,), -7, dtype=torch.int64, device="cuda")
            _h().hash_tokens(dev(flat), 1, token_offsets=dev(toff), seed=7, keys=keys, key_offsets=dev(woff))
            sync()
            got = host(keys, np.int64)
            assert (got[:len(want)] == want).all() and (got[len(want):] == -7).all(), (length, spread)


@pytest.mark.parametrize("general_loader", [False, True])
@pytest.mark.parametrize("dtype,bs,R,lengths", [
    (np.int64, 16, 2048 + 9, (1024, 2048 + 70)),                      # spread: short workgroups direct, long ones staged
    (np.int64, 16, 8192 + 9, (639, 640, 1040)),                       # direct and burst
    (np.int64, 8, 2048 + 9, (511, 512)), (np.int64, 32, 8192 + 9, (895, 900)), (np.int64, 64, 8192 + 9, (895, 897)),
    (np.int64, 128, 4096 + 9, (959, 961)), (np.int64, 1, 33, (63, 200, 513, 1000)), (np.int64, 1, 1100, (512, 513)),
    (np.int32, 8, 12288 + 9, (1279, 1280)), (np.int32, 16, 12288 + 9, (1791, 1800)), (np.int32, 32, 12288 + 9, (1791, 1792)),
    (np.int32, 64, 12288 + 9, (2303, 2304)), (np.int32, 128, 12288 + 9, (2559, 2560)), (np.int32, 1, 64 + 9, (128, 129))])
def test_equally_long_requests_in_every_form_of_the_kernel(oracle, force_general_hash_loader, general_loader, dtype, bs, R, lengths):
    """[R, L] batches on both sides of every line of the launch rule, so that the direct, spread, burst and raw-tile forms all
    read no offset arrays: key offsets written by the launch, or the caller's with gaps between the requests. The last workgroup
    is partial."""
    force_general_hash_loader(general_loader)
    rng = np.random.default_rng(bs + R)
    for L in lengths:
        tok = rng.integers(-2**31, 2**31, size=(R, L), dtype=np.int64).astype(dtype)
        want, woff = oracle.hash_tokens(tok, bs, seed=9, threads=8)
        per = L // bs
        print(f"equally long: {R} x {L} {np.dtype(dtype).name}, block size {bs}", flush=True)
        d_tok = dev(tok)
        keys, off = _h().hash_tokens(d_tok, bs, seed=9)
        sync()
        assert (host(keys, np.int64) == want).all() and (host(off, np.int64) == woff).all(), L
        gaps = np.arange(R + 1, dtype=np.int64) * (per + 1) + 1
        spread = torch.full((R * (per + 1) + 1,), -7, dtype=torch.int64, device="cuda")
        _, same = _h().hash_tokens(d_tok, bs, seed=9, keys=spread, key_offsets=dev(gaps))
        sync()
        got = host(spread, np.int64)
        assert got[0] == -7 and (host(same, np.int64) == gaps).all()
        got = got[1:].reshape(R, per + 1)
        assert (got[:, :per] == want.reshape(R, per)).all() and (got[:, per] == -7).all(), L


@pytest.mark.parametrize("dtype,length", [(np.int64, 4096), (np.int64, 8192), (np.int32, 8192)])
@pytest.mark.parametrize("R", [240 * 64, 240 * 64 - 64])
def test_chains_that_start_32_kib_apart(oracle, dtype, length, R):
    """Block size 1, a workgroup on every CU, requests that start whole multiples of 32 KiB apart: loaders wait for their tokens
    before they write keys. Workgroups where that holds, where one odd request ends it, and where nothing is to do."""
    rng = np.random.default_rng(R)
    lens = np.zeros(R, dtype=np.int64)
    lens[::16] = length                                     # four to a workgroup, the others empty
    lens[64 * 100 + 5] = 77                                 # from here on nobody starts at a multiple ...
    lens[64 * 150 + 5] = length - 77                        # ... and from here on everybody does again
    lens[64 * 200:64 * 201] = 0
    toff = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    flat = rng.integers(-2**31, 2**31, size=int(toff[-1]), dtype=np.int64).astype(dtype)
    want, woff = oracle.hash_tokens(flat, 1, token_offsets=toff, seed=3, threads=8)
    print(f"chains 32 KiB apart: {R} x {length} {np.dtype(dtype).name}", flush=True)
    keys = torch.full((len(want) + 64,), -7, dtype=torch.int64, device="cuda")
    _h().hash_tokens(dev(flat), 1, token_offsets=dev(toff), seed=3, keys=keys, key_offsets=dev(woff))
    sync()
    got = host(keys, np.int64)
    assert (got[:len(want)] == want).all() and (got[len(want):] == -7).all()


@pytest.mark.parametrize("general_loader", [False, True])
@pytest.mark.parametrize("dtype", [np.int64, np.int32])
@pytest.mark.parametrize("bs", [1, 2, 7, 8, 16, 24, 48, 63, 64, 65, 80, 128, 208, 1000])
def test_sixteen_requests_per_workgroup(oracle, force_general_hash_loader, general_loader, dtype, bs):
    """Launches of up to 4096 requests: lengths on and around a tile of 64 tokens, its halves and the 16 steps between two kept
    states, blocks shorter and longer than each of them, workgroups in which one request outlasts the others by many tiles,
    request counts around a workgroup's 16 and around the last count that takes this form; ragged with gaps between the keys of
    neighbours, and equally long."""
    force_general_hash_loader(general_loader)
    rng = np.random.default_rng(bs)
    menu = np.array([0, 1, 15, 16, 17, 31, 32, 33, 47, 48, 63, 64, 65, 95, 96, 97, 127, 128, 129, 191, 192, 193, 255, 256, 257, 320,
                     bs - 1, bs, bs + 1, 2 * bs, 3 * bs + 1])
    for R in (1, 15, 16, 17, 33, 4095, 4096, 4097):
        lens = menu[rng.integers(0, len(menu), size=R)]
        lens[-1] = 1100 if R < 100 else 700                                # the last workgroup outlasts the others
        toff = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
        flat = rng.integers(-2**31, 2**31, size=int(toff[-1]), dtype=np.int64).astype(dtype)
        want, woff = oracle.hash_tokens(flat, bs, token_offsets=toff, seed=R, threads=8)
        koff = woff + np.arange(R + 1)                                      # one slot between neighbours that must stay
        room = torch.full((len(want) + R + 1,), -7, dtype=torch.int64, device="cuda")
        _h().hash_tokens(dev(flat), bs, token_offsets=dev(toff), seed=R, keys=room, key_offsets=dev(koff))
        sync()
        expect = np.full(len(want) + R + 1, -7, dtype=np.int64)
        expect[np.arange(len(want)) + np.repeat(np.arange(R), np.diff(woff))] = want
        assert (host(room, np.int64) == expect).all(), (R, bs)
    for R, L in ((1, 64), (5, 65), (16, 128), (18, 1000), (33, 4096), (4096, 72)):
        tok = rng.integers(-2**31, 2**31, size=(R, L), dtype=np.int64).astype(dtype)
        want, woff = oracle.hash_tokens(tok, bs, seed=-1, threads=8)
        keys, off = _h().hash_tokens(dev(tok), bs, seed=-1)
        sync()
        assert (host(keys, np.int64) == want).all() and (host(off, np.int64) == woff).all(), (R, L, bs)


def _ms(call):
    """The shortest of five runs, in ms of the GPU."""
    best = []
    for _ in range(5):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        call()
        end.record()
        sync()
        best.append(start.elapsed_time(end))
    return min(best)


def test_one_request_of_more_than_a_sixteenth_of_4_gib(oracle):
    """The requests that a workgroup does not have say nothing about how far its tokens reach: one request of 2^28 bytes and more takes
    the loader that keeps up with the chain, at the pace of a shorter one."""
    L = (1 << 25) + 64
    tok = torch.randint(0, 128256, (1, L), dtype=torch.int64, device="cuda")
    keys = torch.empty(L // 4096, dtype=torch.int64, device="cuda")
    short = _ms(lambda: _h().hash_tokens(tok[:, :L // 2].contiguous(), 4096, keys=keys))
    whole = _ms(lambda: _h().hash_tokens(tok, 4096, keys=keys))
    print(f"2^24 tokens {short:.1f} ms, 2^25 {whole:.1f} ms", flush=True)
    want, _ = oracle.hash_tokens(tok.cpu().numpy(), 4096)
    assert (host(keys, np.int64) == want).all()
    assert whole < 2.4 * short


@pytest.mark.parametrize("R", [16, 40])
def test_a_workgroup_of_requests_that_are_left_out_does_not_run(oracle, R):
    """[R, L] batches with the caller's own key offsets, negative for requests whose keys nobody wants: where that is all of a
    workgroup, it takes the time of a launch and not that of the recurrence; the others' keys are where they should be."""
    L = 1 << 16
    tok = torch.randint(0, 128256, (R, L), dtype=torch.int64, device="cuda")
    keys = torch.full((R * (L // 64) + 1,), -7, dtype=torch.int64, device="cuda")
    want, woff = oracle.hash_tokens(tok.cpu().numpy(), 64, threads=8)
    none = torch.full((R + 1,), -1, dtype=torch.int64, device="cuda")
    some = woff.copy()
    some[[0, 5, R - 1]] = -1
    some = dev(some)
    assert _ms(lambda: _h().hash_tokens(tok, 64, keys=keys, key_offsets=none)) < 0.25    # 65 536 steps take 0.7 ms
    assert (host(keys, np.int64) == -7).all()
    _h().hash_tokens(tok, 64, keys=keys, key_offsets=some)
    sync()
    expect = want.reshape(R, -1).copy()
    expect[[0, 5, R - 1]] = -7
    assert (host(keys, np.int64)[:-1] == expect.reshape(-1)).all()


def test_hash_strings_that_wait_behind_other_work(monkeypatch):
    """Calls whose strings the kernel has yet to read when the next ones arrive: more of them than are read in place, from two
    threads, strings of many lengths; then more bytes than are read in place; and nothing stays lent out."""
    import threading
    h = _h()
    monkeypatch.setattr(h, "_LENT_MOST", 8)

    def key(s):
        return int.from_bytes(hashlib.sha256(s.encode()).digest()[:8], "big", signed=True)

    got = {}

    def many(t):
        torch.cuda._sleep(2_000_000)
        for i in range(20):
            strs = [chr(97 + (i + k) % 26) * ((7 * i + 13 * k + t) % 140) for k in range(1 + 11 * i)]
            got[t, i] = (strs, h.sha256_to_int64(strs))

    threads = [threading.Thread(target=many, args=(t,)) for t in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    sync()
    assert len(got) == 40
    for strs, keys in got.values():
        assert keys.tolist() == [key(s) for s in strs]
    monkeypatch.setattr(h, "_PINNED_MOST", 100)
    assert h.sha256_to_int64(["x" * 200, "y"]).tolist() == [key("x" * 200), key("y")]
    monkeypatch.undo()
    h.sha256_to_int64(["z"])
    sync()
    assert h._settled_event(torch.device("cuda:0")) is not None and not h._lent
