"""Snapshot import decoded on the device (kv_cbor_decode_device) against the
strict host reader, on the same documents.

Every document is imported twice: as it is (64 KiB or more in the encoder's own
form: decoded on the device), and with an unknown field put first in its top
map, which serde skips and only the strict reader accepts.  Both must give the
same rows bit for bit, or fail with the same message."""
import struct

import numpy as np
import pytest

import oracle as O
from mesh_amd import DeviceContext, KVCacheBlob, KVCacheWireSnapshot, KVSequenceState, ModelGeometry
from mesh_amd._lib import ZrError

pytestmark = pytest.mark.gpu

LAYERS, KV_HEADS, D = 2, 4, 64
COLS = KV_HEADS * D


@pytest.fixture(scope="module")
def ctx():
    geo = ModelGeometry(hidden=D * 8, num_heads=8, num_kv_heads=KV_HEADS, num_layers=LAYERS, vocab=64, ffn=64)
    c = DeviceContext(geo, kv_dtype="f32", max_tokens=64, max_seqs=4, max_pages_per_seq=200)
    c.create_kv_pool(400)
    yield c
    c.close()


def outcome(ctx, doc, rows, nxt):
    b = ctx.new_backend(4096)
    try:
        b.import_kv_snapshot(KVCacheWireSnapshot(KVSequenceState(nxt, rows),
                                                 KVCacheBlob("FullSnapshotCbor", memoryview(bytes(doc)))))
        snap = b.export_kv_cache()
        return "rows", snap.keys.view(np.uint32).tobytes() + snap.values.view(np.uint32).tobytes()
    except ZrError as e:
        assert b.cache_seq_len() == 0
        return "error", str(e)
    finally:
        b.release_pages()
        b.close()


def check(ctx, doc, rows, nxt, expect=None):
    doc = bytes(doc)
    got = outcome(ctx, doc, rows, nxt)
    assert got == outcome(ctx, b"\xa4\x61x\x00" + doc[1:], rows, nxt)
    if expect:
        assert got[0] == expect, got
    return got


def document(rows, seed, nxt, kind="mixed"):
    rng = np.random.default_rng(seed)
    kv = rng.standard_normal((2, LAYERS, rows, COLS)).astype(np.float32)
    if kind == "halves":
        kv = kv.astype(np.float16).astype(np.float32)
    elif kind == "mixed":  # 3- and 5-byte items in no pattern; bytes that look like heads inside the singles
        half = rng.random(kv.shape) < 0.5
        kv = np.where(half, kv.astype(np.float16).astype(np.float32), kv)
        odd = rng.random(kv.shape) < 0.05
        bits = rng.choice(np.array([0xF9FAFBF9, 0xFAFAFAFA, 0x7BFBFBFB, 0x1B1A1918, 0x6D6D6D6D], np.uint32), kv.shape)
        kv = np.where(odd, bits.view(np.float32), kv)
        kv.reshape(-1)[:8] = [0.0, -0.0, np.inf, -np.inf, 2.0 ** -24, 1e-40, 65504.0, 2.0 ** -14]
    return kv, O.kv_cbor_encode(kv[0], kv[1], nxt - rows, LAYERS, KV_HEADS, D, 4096)


@pytest.mark.parametrize("kind", ["halves", "singles", "mixed"])
@pytest.mark.parametrize("rows,ahead", [(13, 0), (33, 7), (64, 300), (171, 70000), (1000, 1)])
def test_documents_of_every_size_decode_to_their_rows(ctx, kind, rows, ahead):
    """Below the size line and above it, over one to dozens of 16 KiB blocks,
    base positions with 1- to 5-byte integers."""
    kv, doc = document(rows, rows + ahead, rows + ahead, kind)
    _, got = check(ctx, doc, rows, rows + ahead, "rows")
    assert got == kv.view(np.uint32).tobytes()


def test_double_items_round_as_the_strict_reader(ctx):
    """9-byte items: finite values (rounded to f32), f32 subnormals, overflow, NaN payloads."""
    rows = 40
    kv, doc = document(rows, 5, rows, "halves")
    rng = np.random.default_rng(6)
    doubles = np.concatenate([rng.standard_normal(200), rng.standard_normal(50) * 1e-41, rng.standard_normal(20) * 1e300,
                              [0.0, -0.0, np.inf, -np.inf, 1e-320]]).astype(np.float64)
    raw = [struct.pack(">d", x) for x in doubles]
    raw += [struct.pack(">Q", q) for q in (0x7FF8000000000000, 0xFFF0000000000001, 0x7FF4000020000001, 0x7FFFFFFFFFFFFFFF)]
    at = doc.index(b"ddata") + 8  # 0x99 and two length bytes: 40 x 256 floats
    assert doc[at - 3] == 0x99 and doc[at] == 0xF9
    head, tail = doc[:at], doc[at + 3 * len(raw):]
    check(ctx, head + b"".join(b"\xfb" + r for r in raw) + tail, rows, rows, "rows")


@pytest.mark.parametrize("seed", range(6))
def test_damaged_documents_end_as_with_the_strict_reader(ctx, seed):
    """Truncation, trailing bytes, a changed byte anywhere, an integer of the
    same size in place of a float, an item removed or doubled, another key."""
    rows = 60
    _, doc = document(rows, 100 + seed, rows, ["mixed", "halves"][seed % 2])
    rng = np.random.default_rng(seed)
    at = doc.index(b"ddata") + 8
    check(ctx, doc[:-1], rows, rows, "error")
    check(ctx, doc + b"\xf9\x00\x00", rows, rows, "error")
    check(ctx, doc[:len(doc) // 2], rows, rows, "error")
    for p in list(rng.integers(1, len(doc), 12)) + [1, 2, at, at - 1, len(doc) - 2]:
        x = bytearray(doc)
        x[p] = int(rng.integers(0, 256))
        check(ctx, x, rows, rows)
    if doc[at] == 0xF9:
        check(ctx, doc[:at] + b"\x19\x01\x02" + doc[at + 3:], rows, rows, "error")
        check(ctx, doc[:at] + doc[at + 3:], rows, rows, "error")
        check(ctx, doc[:at] + doc[at:at + 3] * 2 + doc[at + 3:], rows, rows, "error")
        # one float fewer and an integer more: as many items, no float array
        check(ctx, doc[:at] + b"\x00\x00\x00" + doc[at + 3:], rows, rows, "error")
    p = doc.rindex(b"gseq_len")
    check(ctx, doc[:p] + b"gseq_lem" + doc[p + 8:], rows, rows, "error")
    check(ctx, doc.replace(b"jnum_layers", b"jnum_lawers"), rows, rows, "rows")  # an unknown config key is skipped
    check(ctx, doc, rows, rows + 1, "error")
    check(ctx, doc, rows - 1, rows, "error")
    check(ctx, doc, rows, rows, "rows")


def test_other_forms_of_the_document_still_import(ctx):
    """Longer integers than needed, fields in another order: the strict reader's."""
    rows = 50
    kv, doc = document(rows, 9, rows, "halves")
    want = kv.view(np.uint32).tobytes()
    p = doc.rindex(b"mbase_position")
    assert doc[p + 14] == 0
    assert check(ctx, doc[:p + 14] + b"\x18\x00" + doc[p + 15:], rows, rows, "rows")[1] == want
    end = doc[p:]
    moved = b"\xa3" + end + doc[1:p]
    assert check(ctx, moved, rows, rows, "rows")[1] == want


def test_small_rows_and_a_full_pool(ctx):
    """Few columns per layer stay with the strict reader; a pool without room fails as before and changes nothing."""
    geo = ModelGeometry(hidden=64, num_heads=4, num_kv_heads=1, num_layers=2, vocab=64, ffn=64)
    c = DeviceContext(geo, kv_dtype="f32", max_tokens=16, max_seqs=2, max_pages_per_seq=400)
    c.create_kv_pool(300)
    rows = 3000
    k = np.random.default_rng(1).standard_normal((2, 2, rows, 16)).astype(np.float32)
    doc = O.kv_cbor_encode(k[0], k[1], 0, 2, 1, 16, 4096)
    assert check(c, doc, rows, rows, "rows")[1] == k.view(np.uint32).tobytes()
    c.create_kv_pool(20)
    free = c.free_pages
    assert "error" == check(c, doc, rows, rows)[0]
    assert c.free_pages == free
    c.close()
