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
