"""The persistent traversal's grids on a runtime without a device: every instance of the kernel
is launched with the workgroups that this instance keeps resident. A row dealt to a workgroup
that is not resident waits until the others have drained the rest of the queue."""
import os
import re
import sys

import pytest

sys.path[:0] = [os.path.dirname(os.path.abspath(__file__)),
                os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pbr-rust_amd")]
import fake_hip  # noqa: E402

CUS = 256


def instance(kernel):
    """(multi, flags) of a traversal kernel's mangled name, None for other kernels."""
    m = re.search(r"trace_wide_(multi_)?kernelI((?:Lb[01]E)+)E", kernel)
    return m and (bool(m.group(1)), re.findall(r"Lb([01])E", m.group(2)))


def occupancy(kernel):
    """A number of its own for every instance."""
    inst = instance(kernel)
    return 1 if inst is None else 2 + int(inst[0]) * 4 + int("".join(inst[1]), 2)


def grids(shapes, kind):
    seen = {}

    def launch(kernel, blocks, threads, captured, args):
        if instance(kernel):
            seen.setdefault(kernel, set()).add(blocks)
        elif "round_end_multi" in kernel:
            fake_hip.poke_u32(fake_hip.pointer(args, 0) + 8, 1)  # the batch is over

    fake_hip.install(launch, occupancy=occupancy)
    import pbrtm
    from pbrtm import scenes

    with pbrtm.Context(0) as ctx:
        # 2^20 slots: more rows than any grid here has waves
        scene = ctx.scene((scenes.shapes_room if shapes == "shapes" else scenes.cornell34)(512, 512))
        if kind == "batch":
            ctx.render_batch([(scene, 4, 3, 0)], graph=False)
        else:
            scene.render(spp=4, max_depth=3, count=kind == "count")
        scene.free()
    assert len(seen) == 1, seen
    (kernel, blocks), = seen.items()
    multi, flags = instance(kernel)
    assert multi == (kind == "batch") and flags[-1] == str(int(shapes == "shapes"))
    assert multi or flags[0] == str(int(kind == "count"))
    assert blocks == {occupancy(kernel) * CUS}, (kernel, blocks)


@fake_hip.needs_compiler
@pytest.mark.parametrize("kind", ["render", "count", "batch"])
@pytest.mark.parametrize("shapes", ["triangles", "shapes"])
def test_grid_of_each_instance(tmp_path, shapes, kind):
    fake_hip.isolated(__file__, "grids", tmp_path, shapes, kind)


if __name__ == "__main__":
    fake_hip.main(globals())
