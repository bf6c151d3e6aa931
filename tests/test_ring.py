"""The product's ring bookkeeping (gh_ring_*) against the oracle's
restatement of src/ring_buffer.zig and the reference's own ring tests."""
import numpy as np

import gemma_hip as gh
import oracle as orc


def test_ring_reference_kat_window_eviction():
    # src/ring_buffer.zig:149-166
    r = gh.Ring(2, 4, 8, 4)
    assert r.total_slots == 16
    for c in range(20):
        r.activate_slot(0, c)
    s = r.active_slots(0, 19)
    assert len(s) == 12 and s[0] == 0 and s[3] == 3


def test_ring_reference_kat_recall():
    # src/ring_buffer.zig:168-187
    r = gh.Ring(1, 2, 4, 3)
    r.activate_recall(0, 0, 100)
    r.activate_recall(0, 1, 50)
    assert len(r.active_slots(0, 101)) == 2
    r.clear_recall()
    assert len(r.active_slots(0, 101)) == 0


def test_ring_matches_oracle_random():
    rng = np.random.default_rng(12)
    for A, W, R in [(32, 512, 96), (4, 16, 4), (0, 8, 2), (3, 5, 0)]:
        g = gh.Ring(2, A, W, R)
        o = orc.Ring(2, 1, A, W, R)
        clock = 0
        for step in range(700):
            clock += int(rng.integers(1, 3))
            for layer in (0, 1):
                assert g.activate_slot(layer, clock) == o.activate_slot(layer, clock)
            if R and rng.random() < 0.05:
                rank = int(rng.integers(0, R))
                c = int(rng.integers(0, clock + 20))
                g.activate_recall(0, rank, c)
                o.write_recall_kv(0, rank, np.zeros(1, np.float32), np.zeros(1, np.float32), c)
            if R and rng.random() < 0.02:
                g.clear_recall()
                o.clear_recall()
            q = clock + int(rng.integers(-3, 3))
            q = max(q, 0)
            assert np.array_equal(g.active_slots(0, q), o.active_slots(0, q))
            assert g.slot_index(q) == o.slot_index(q)


def test_ring_lists_by_room():
    """Lists cut by the caller's room: the first `cap` entries of the whole
    list, its full length returned, nothing written past the room; over rings
    whose tiers are no multiple of eight and windows that are empty in part."""
    rng = np.random.default_rng(7)
    for A, W, R in [(32, 512, 96), (3, 13, 5), (0, 24, 0), (9, 8, 1)]:
        for filled in (0, 1, W // 2, W + A):
            g = gh.Ring(1, A, W, R)
            o = orc.Ring(1, 1, A, W, R)
            for c in range(filled):
                if rng.random() < 0.8:
                    g.activate_slot(0, c)
                    o.activate_slot(0, c)
            for rank in range(0, R, 3):
                c = int(rng.integers(0, 2 * W))
                g.activate_recall(0, rank, c)
                o.write_recall_kv(0, rank, np.zeros(1, np.float32), np.zeros(1, np.float32), c)
            for q in (0, filled // 2, max(filled - 1, 0), filled + W // 2):
                want = o.active_slots(0, q)
                for cap in (0, 1, 7, 8, 9, len(want), g.total_slots):
                    out = np.full(cap + 8, 0xFFFFFFFF, np.uint32)
                    n = gh.lib().gh_ring_active_slots(g.h, 0, q, gh._ptr(out), cap)
                    assert n == len(want)
                    assert np.array_equal(out[:min(n, cap)], want[:cap])
                    assert (out[cap:] == 0xFFFFFFFF).all()


def test_ring_lists_leave_the_room_behind_them():
    """Room past the list's end keeps what it held: a host may pack lists one
    behind another, or keep words of its own there."""
    rng = np.random.default_rng(8)
    for A, W, R in [(32, 512, 96), (3, 13, 5), (0, 24, 0), (9, 8, 1), (2, 16, 8)]:
        g = gh.Ring(1, A, W, R)
        for c in range(2 * W):
            if rng.random() < 0.7:
                g.activate_slot(0, c)
            if R and rng.random() < 0.2:
                g.activate_recall(0, int(rng.integers(0, R)), int(rng.integers(0, 2 * W)))
            q = int(rng.integers(0, c + 2))
            want = g.active_slots(0, q)
            out = np.full(g.total_slots + 16, 0xFFFFFFFF, np.uint32)
            n = gh.lib().gh_ring_active_slots(g.h, 0, q, gh._ptr(out), len(out))
            assert n == len(want) and np.array_equal(out[:n], want)
            assert (out[n:] == 0xFFFFFFFF).all()
