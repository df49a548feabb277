"""The rollout's replay: the backward linearises about the forward's own states,
so replaying an interval from its checkpoint, unfused and with records, must end
at the next checkpoint bit for bit, also with boundary data that depend on time
and whose steps' times round differently from start and checkpoint."""
import numpy as np
import pytest

from helpers import grids

pytestmark = pytest.mark.gpu

mif = pytest.importorskip("mif_amd")
torch = pytest.importorskip("torch")

from mif_amd.autograd import Rollout  # noqa: E402

STEPS, EVERY = 14, 5


def rollout(Ng, per, form, kind):
    _, gs = grids(Ng, (1.0, 1.0, 2.0), (0.0, 0.0, -1.0), 1e2, STEPS * 1.1e-3, STEPS, per)
    ctx = mif.Context(gs, precision=mif.FP64 if form == "fp64" else mif.MIXED)
    roll = Rollout(ctx, STEPS, checkpoint_every=EVERY, exact_velocity=mif.function(kind, Re=1e2))
    rng = np.random.default_rng(5)
    return ctx, roll, [torch.tensor(0.1 * rng.standard_normal(s), device="cuda") for s in roll.shapes]


@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("Ng,per,kind", [((17, 20, 19), (0, 0, 0), "VT_VELOCITY"), ((33, 18, 25), (1, 0, 1), "ZERO"),
                                         ((65, 70, 66), (1, 0, 1), "VT_VELOCITY"), ((67, 66, 61), (0, 0, 0), "LID_1")])
def test_replay_ends_at_the_next_checkpoint(Ng, per, kind, form):
    print(f"[case] rollout replay {form} {Ng} periodic={per} {kind}", flush=True)
    ctx, roll, u0 = rollout(Ng, per, form, getattr(mif, "FN_" + kind))
    assert any(s * ctx.dt != EVERY * ctx.dt + (s - EVERY) * ctx.dt for s in range(EVERY, 2 * EVERY))
    roll.run_forward(u0, (0.02, 0.0, -0.01))
    for c in range(len(roll.cp_u) - 1):
        roll.vel.copy_from(roll.cp_u[c])
        roll.p.copy_from(roll.cp_p[c])
        for s in range(c * EVERY, (c + 1) * EVERY):
            roll._record_step(s, c * EVERY)
        for a, b in zip([*roll.vel.download(), roll.p.download()],
                        [*roll.cp_u[c + 1].download(), roll.cp_p[c + 1].download()]):
            assert np.array_equal(a, b)
    ctx.close()


def test_the_context_keeps_its_own_records_setting():
    """A context that other steps use with fused projections keeps them so, and
    the rollout's gradient does not depend on the setting."""
    print("[case] rollout leaves the stage records setting", flush=True)
    grads, fields = [], []
    for keep in (True, False):
        ctx, roll, u0 = rollout((17, 20, 19), (0, 0, 0), "fp64", mif.FN_ZERO)
        ctx.set_stage_records(keep)
        us = [t.clone().requires_grad_(True) for t in u0]
        f = torch.zeros(3, dtype=torch.float64, requires_grad=True)
        out = roll(us, f)
        grads.append(torch.autograd.grad(sum((t * t).sum() for t in out), [*us, f]))
        vel, buf, buf2, p, pb = ctx.velocity(), ctx.velocity(), ctx.velocity(), ctx.pressure(), ctx.pressure()
        vel.upload([t.cpu().numpy() for t in u0])
        mif.timestep(vel, buf, buf2, roll.ev, 0.0, p, pb)
        fields.append(buf.download())
        if not keep:  # what a context without a rollout leaves in its buffer
            fresh = mif.Context(ctx.grid)
            v, b, b2, q, qb = (fresh.velocity(), fresh.velocity(), fresh.velocity(), fresh.pressure(),
                               fresh.pressure())
            v.upload([t.cpu().numpy() for t in u0])
            mif.timestep(v, b, b2, roll.ev, 0.0, q, qb)
            for x, y in zip(buf.download(), b.download()):
                assert np.array_equal(x, y)
            fresh.close()
        ctx.close()
    for a, b in zip(*grads):
        assert torch.equal(a, b)
    assert not np.array_equal(fields[0][0], fields[1][0])
