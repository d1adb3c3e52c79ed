"""GatherPlan as callers hold it: its method by keyword, overridden, kept without the plan, and a plan
for no windows."""
import pytest

from conftest import announce

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _plan(cls, num, table):
    dst = torch.empty(num, 8, dtype=torch.uint8, device="cuda")
    return cls(table, 64, [dict(dst=dst, ofst=0, span=2, step_bytes=4, col_base=0, pad_head=False)],
               num), dst


def _args(num):
    return dict(idxs=torch.arange(num, device="cuda"),
                tss=torch.zeros(num, dtype=torch.int64, device="cuda"),
                lens=torch.full((num,), 16, dtype=torch.int64, device="cuda"))


def test_run_by_keyword_and_overridden():
    from gear_amd import ops
    table = torch.randint(0, 255, (64 * 5,), dtype=torch.uint8, device="cuda")

    class Counted(ops.GatherPlan):
        calls = 0

        def run(self, idxs, tss, lens):
            self.calls += 1
            return super().run(idxs, tss, lens)

    announce("gather plan by keyword")
    for cls in (ops.GatherPlan, Counted):
        plan, dst = _plan(cls, 5, table)
        plan.run(**_args(5))
        plan.run(lens=_args(5)["lens"], idxs=_args(5)["idxs"], tss=_args(5)["tss"])
        assert torch.equal(dst, table.view(5, 64)[:, :8])
    assert plan.calls == 2


def test_the_method_keeps_its_tensors():
    import gc
    import weakref
    from gear_amd import ops
    announce("gather plan kept by its method")
    table = torch.zeros(64 * 3, dtype=torch.uint8, device="cuda")
    plan, dst = _plan(ops.GatherPlan, 3, table)
    alive = [weakref.ref(table), weakref.ref(dst)]
    run = plan.run
    del plan, table, dst
    gc.collect()
    assert all(r() is not None for r in alive)
    run(**_args(3))
    torch.cuda.synchronize()


def test_a_plan_for_no_windows():
    from gear_amd import ops
    announce("gather plan of no windows")
    plan, dst = _plan(ops.GatherPlan, 0, torch.zeros(64, dtype=torch.uint8, device="cuda"))
    plan.run(**_args(0))
    with pytest.raises(ValueError, match="made for 0 windows"):
        plan.run(**_args(1))
