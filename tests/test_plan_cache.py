"""The plans an operator keeps, used by several threads at once (no GPU involved)."""
import threading

from sparsetir_amd.ops import _PlanCache


class _Key:
    """A key whose second hash after ``armed`` is set lets another thread run first."""

    def __init__(self, other):
        self.other, self.armed, self.asked = other, False, 0

    def __hash__(self):
        self.asked += self.armed
        if self.armed and self.asked == 2:
            self.armed = False
            self.other()
        return 7

    def __eq__(self, o):
        return self is o


def test_a_plan_found_is_not_destroyed_by_another_thread():
    """Between looking a plan up and moving it to the front, another thread wants to fill the cache: it waits."""
    destroyed = []
    cache = _PlanCache(destroyed.append, lambda name: None)

    def fill():
        for k in range(cache.capacity):
            cache.put(("other", k), f"plan {k}", None)

    thread = threading.Thread(target=fill)

    def other():
        thread.start()
        thread.join(0.3)

    key = _Key(other)
    cache.put(key, "mine", None)
    cache.put("later", "later", None)
    key.armed = True
    assert cache.get(key) == "mine"
    thread.join()
    assert destroyed == ["later", "mine"] and len(cache) == cache.capacity


def test_forget_comes_before_destroy():
    """The launcher has let go of a plan before it is destroyed."""
    log = []
    cache = _PlanCache(lambda plan: log.append(("destroy", plan)), lambda name: log.append(("forget", name)))
    for k in range(cache.capacity + 1):
        cache.put(k, f"p{k}", None)
    assert log == [("forget", 0), ("destroy", "p0")]
    cache.clear()
    assert log[2] == ("forget", None) and len(log) == 3 + cache.capacity and len(cache) == 0
