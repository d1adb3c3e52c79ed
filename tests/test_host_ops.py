"""Argument checks of gear_amd.ops (made natively): refused before anything reaches the GPU, with
the name of the argument."""
import pytest

torch = pytest.importorskip("torch")


def test_wrong_arguments_are_named():
    from gear_amd import ops
    f = torch.zeros(8)
    with pytest.raises(TypeError, match="priorities must be a torch.Tensor"):
        ops.prefix_sum([1.0, 2.0])
    with pytest.raises(TypeError, match="priorities must have dtype torch.float32, got torch.float64"):
        ops.prefix_sum(f.double())
    with pytest.raises(ValueError, match="priorities must be contiguous"):
        ops.prefix_sum(f[::2])
    with pytest.raises(ValueError, match="priorities must live on the GPU"):
        ops.prefix_sum(f)
    with pytest.raises(TypeError, match="weights must have dtype torch.int64"):
        ops.prefix_sum_i64(f)
    with pytest.raises(TypeError, match="prefix must have dtype torch.float64"):
        ops.upper_bound(f, f)
    with pytest.raises(TypeError, match="prefix must have dtype torch.float64"):
        ops.sample_sorted(f, f)
    with pytest.raises(ValueError, match="window starts come with an int64 prefix only"):
        ops.sample_lookup(f.double(), f, start_uniforms=f.double(), window=2)
    with pytest.raises(TypeError, match="positions must have dtype torch.int64"):
        ops.sort_lookup(f, 8)
    with pytest.raises(TypeError, match="keys must have dtype torch.int64"):
        ops.sort_i64(f)
    with pytest.raises(TypeError, match="scatter works on float32 or int64 tables"):
        ops.scatter(f.double(), f.long(), f.double())


def test_a_number_of_entries_is_an_integer():
    """Integers of any type count, a fraction is refused and not cut off."""
    import numpy as np
    from gear_amd import ops
    f = torch.zeros(8)
    for k in (2, np.int64(2), torch.tensor(2)):
        with pytest.raises(ValueError, match="priorities must live on the GPU"):
            ops.topk(f, k)
    for k in (2.0, 2.7, "2", None):
        with pytest.raises(TypeError):
            ops.topk(f, k)


@pytest.mark.parametrize("name", ["draw", "prepare"])
@pytest.mark.parametrize("where", ["class", "sampler", "subclass"])
def test_replaced_draws_are_asked_for(monkeypatch, name, where):
    """A loader's step draws by itself only where draw() and prepare() are the sampler's own."""
    from gear_amd.mpu import ModelParallelismUnit
    from gear_amd.sampler import UniformSampler, WeightedSampler
    mpu = ModelParallelismUnit(device=torch.device("cpu"))
    for cls in (UniformSampler, WeightedSampler):
        sampler = cls(mpu)
        assert sampler.draws_of_a_step(10, 4) is sampler._generator
        called = []

        def draw(*a, **kw):
            called.append(a)
            return torch.zeros(4)

        with monkeypatch.context() as m:
            if where == "sampler":
                m.setattr(sampler, name, draw, raising=False)
            elif where == "class":
                m.setattr(cls, name, draw)
            else:
                sampler = type("Own", (cls,), {name: draw})(mpu)
            assert isinstance(sampler.draws_of_a_step(10, 4), torch.Tensor)
            assert len(called) == (name == "draw")
