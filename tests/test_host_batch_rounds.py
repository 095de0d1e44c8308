"""pbrtm_render_batch's rounds per launch over the whole range of the parameter, on a runtime
without a device: every call ends, and holds a bounded number of rounds in a launch."""
import os
import sys

import pytest

sys.path[:0] = [os.path.dirname(os.path.abspath(__file__)),
                os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pbr-rust_amd")]
import fake_hip  # noqa: E402

K_DONE = 2  # counter word: the batch is over
MAX_ROUNDS = 1024


def batch(rpl, graph):
    """One batch of two jobs; its rounds (their last kernel) are counted, and the first launch
    that holds a round ends the batch."""
    rpl, graph = int(rpl), graph == "graph"
    seen = {"rounds": 0, "launches": 0, "counters": 0}

    def launch(kernel, blocks, threads, captured, args):
        if "round_end_multi" not in kernel:
            return 0
        assert captured == graph
        seen["rounds"] += 1
        seen["counters"] = fake_hip.pointer(args, 0)
        if not captured:
            fake_hip.poke_u32(seen["counters"] + 4 * K_DONE, 1)
        return 0 if seen["rounds"] <= 4 * MAX_ROUNDS else 1  # a launch without end is refused here

    def graph_launch():
        seen["launches"] += 1
        if seen["rounds"]:
            fake_hip.poke_u32(seen["counters"] + 4 * K_DONE, 1)
        return 0 if seen["launches"] <= 100 else 1

    fake_hip.install(launch, graph_launch)
    import pbrtm
    from pbrtm import scenes

    with pbrtm.Context(0) as ctx:
        jobs = [(ctx.scene(scenes.cornell34(8, 8)), 4, 4000, 0), (ctx.scene(scenes.cornell34(5, 3)), 1, 2, 0)]
        _, _, _, st = ctx.render_batch(jobs, pool_size=1, rounds_per_launch=rpl, graph=graph)
        for scene, *_ in jobs:
            scene.free()
    want = rpl or 8
    assert seen["rounds"] == min(want + want % 2, MAX_ROUNDS), seen  # the queues' parity: an even number
    assert st["launches"] == 1


@fake_hip.needs_compiler
@pytest.mark.parametrize("mode", ["graph", "stream"])
@pytest.mark.parametrize("rpl", [0, 1, 2, 3, 1023, 1024, 1025, 0x7FFFFFFF, 0xFFFFFFFE, 0xFFFFFFFF])
def test_rounds_per_launch(tmp_path, rpl, mode):
    fake_hip.isolated(__file__, "batch", tmp_path, str(rpl), mode)


if __name__ == "__main__":
    fake_hip.main(globals())
