"""Steps taken on the candidates between list builds (deme_step with detection every step and no drift margin) against
the contact-list path (the cell sweep every pass): states, contact lists, persistent maps, histories and records bit for
bit, over what a candidate may meet -- planes that move, masks and families that change on the way, scenes of a batch,
user force models, spheres at the end of the bin grid, lists that go stale or die at once, empty systems -- and over
calls too short to use them."""
import numpy as np
import pytest

from deme_amd import scenes
from deme_amd.abi import ANAL_DTYPE, RULE_DTYPE, DemeError, DeviceSystem

pytestmark = pytest.mark.gpu

LINEAR = """
    const float vn = dot(ALinVel - BLinVel, B2A);
    force = (float)(2e3 * overlapDepth) * B2A - (1.0f * vn) * B2A;
    contact_age += ts;
"""


def _same(a, b):
    sa, sb = a.get_state(), b.get_state()
    for k in sa:
        assert np.array_equal(sa[k], sb[k]), k
    ca, cb = a.counts(), b.counts()
    for k in ("nContacts", "nPrevContacts", "nSphereGeoContacts", "nSteps", "time"):
        assert getattr(ca, k) == getattr(cb, k), k
    for x, y in zip(a.contacts(), b.contacts()):
        assert np.array_equal(x, y)
    assert np.array_equal(a.wildcards(), b.wildcards())


def _pair(sc, setup=None):
    a, b = DeviceSystem(sc), DeviceSystem(sc)
    b.set_skin(0.0)
    for d in (a, b):
        if setup:
            setup(d)
    return a, b


def _clumps_masked():
    sc = scenes.clump_settling(n_clumps=3001, box=(0.1, 0.1, 0.2), velocity_sigma=0.3, omega_sigma=20.0, seed=51)
    fam = np.random.default_rng(1).integers(0, 3, sc.n_clumps)
    sc.state["family"][:sc.n_clumps] = fam
    sc.mask[1 * 2 // 2 + 0] = 1  # families 0 and 1 do not touch
    sc.mask[2 * 3 // 2 + 2] = 1  # nor family 2 among itself
    rule = "if (family_code == 1 && t > 2.4e-4f) newFamily = 2; else if (family_code == 2 && vel.z < -0.4f) newFamily = 0;"
    return sc, lambda d: d.set_motion_rules(family_change_rules=rule)


def _bed_fast_plate():
    sc = scenes.polydisperse_bed(n=9001, seed=52, relax_iters=4, plate_speed=30.0, h=2e-6)
    sc.state["vX"][:sc.n_clumps] = np.random.default_rng(2).normal(0, 0.3, sc.n_clumps)
    return sc, None


def _batch():
    return scenes.batched_columns(n_scenes=7, total_scale=0.02, pitch_scale=0.8, seed=53), None


def _model():
    sc = scenes.sphere_settling(n=4003, spacing=1.98, velocity_sigma=0.3, omega_sigma=5.0, seed=54)

    def setup(d):
        d.set_force_model(LINEAR, ["contact_age"])
        d.keep_contact_records(True)

    return sc, setup


def _rolling():
    return scenes.sphere_settling(n=2500, spacing=1.98, velocity_sigma=0.5, omega_sigma=30.0, Crr=0.05, seed=55), None


def _fast_gas():
    # lists die within a few steps even at the widest automatic skin
    return scenes.sphere_settling(n=2000, spacing=3.0, velocity_sigma=60.0, seed=56), None


def _at_the_grid_end():
    # a box an exact multiple of the bin size, spheres pressed into its upper walls: bin ranges end at the grid's end
    r = 0.005
    L = 0.16
    g = np.stack(np.meshgrid(*[np.arange(15)] * 3, indexing="ij"), -1).reshape(-1, 3) * (2 * r * 0.995)
    g = g - g.max(0) + (L / 2 - 0.98 * r)
    vel = np.random.default_rng(3).normal(0, 0.1, g.shape)
    return scenes.spheres_scene(g, r, (L, L, L), vel=vel), None


def _apart():
    # nothing in contact, no candidates: a grid of distant spheres without planes
    g = np.stack(np.meshgrid(*[np.arange(4)] * 3, indexing="ij"), -1).reshape(-1, 3) * 0.05
    return scenes.spheres_scene(g - g.mean(0), 0.002, (0.4, 0.4, 0.4), planes=False), None


SCENES = {f.__name__[1:]: f for f in (_clumps_masked, _bed_fast_plate, _batch, _model, _rolling, _fast_gas,
                                      _at_the_grid_end, _apart)}


@pytest.mark.parametrize("skin", [None, 3e-5])
@pytest.mark.parametrize("name", sorted(SCENES))
def test_steps_on_the_candidates_equal_the_contact_list_path(name, skin):
    sc, setup = SCENES[name]()
    a, b = _pair(sc, setup)
    if skin is not None:
        a.set_skin(skin)
    done = 0
    for chunk in (1, 5, 6, 7, 40, 1, 70):
        a.step(chunk, 1)
        b.step(chunk, 1)
        _same(a, b)
        if name == "model":
            for x, y in zip(a.forces(), b.forces()):
                assert np.array_equal(x, y)
        # all but the last step of a call of six or more; the gas's lists die at once, so that the automatic skin gives way
        # to the cell sweep before a call is long enough
        now = a.path_stats()[0] - done
        assert now == 0 if chunk < 6 or (name, skin) == ("fast_gas", None) else chunk - 2 <= now <= chunk - 1
        done += now
    assert b.path_stats()[:2] == (0, 0)
    if name not in ("apart",):
        assert a.counts().nContacts > 20


def test_a_plane_turned_into_the_bed_is_met():
    """A fixed plane far from every sphere, rotated between calls by a new state: its spheres are listed anew."""
    sc = scenes.sphere_settling(n=3000, spacing=1.99, velocity_sigma=0.2, seed=57)
    nc = sc.n_clumps
    extra = np.zeros(1, ANAL_DTYPE)
    extra[0]["owner"] = nc + 1
    extra[0]["relPos"] = (0.0, 0.0, -0.29)
    extra[0]["rot"] = (0.0, 0.0, 1.0)
    extra[0]["mass"] = 1e15
    sc.anal = np.concatenate([sc.anal, extra])
    sc.state = {q: np.concatenate([v, v[nc:nc + 1]]) for q, v in sc.state.items()}
    sc.state["family"][nc + 1] = 9
    rule = np.zeros(1, RULE_DTYPE)[0]
    rule["used"] = rule["linVelPrescribed"] = rule["rotVelPrescribed"] = 1
    rule["velSet"] = 0x3F
    rule["vel"][:] = (0.0, 0.0, 0.0, 0.0, 400.0, 0.0)  # turns by 4 mrad a step
    sc.rules[9] = rule
    sc.n_owners = nc + 2
    sc.owner_mass = np.append(sc.owner_mass, np.float32(1e15))
    sc.owner_moi = np.ascontiguousarray(np.append(sc.owner_moi, np.full((1, 3), 1e15, np.float32), 0))
    a, b = _pair(sc)
    for chunk in (10, 30, 25):
        a.step(chunk, 1)
        b.step(chunk, 1)
        _same(a, b)
    st = a.get_state()
    st["oriQw"][nc + 1], st["oriQx"][nc + 1] = np.float32(0.9), np.float32(np.sqrt(1 - 0.81))
    for d in (a, b):
        d.set_state(st)
        d.step(20, 1)
    _same(a, b)


def test_a_sphere_leaving_the_world_fails_at_the_same_step():
    g = np.stack(np.meshgrid(np.arange(6), np.arange(6), np.arange(3), indexing="ij"), -1).reshape(-1, 3) * 0.0098
    xyz = np.concatenate([g - g.mean(0), [[0.0, 0.0, 0.04]]])
    vel = np.zeros_like(xyz)
    vel[-1] = (0.0, 0.0, 100.0)
    sc = scenes.spheres_scene(xyz, 0.005, (0.1295, 0.1295, 0.1295), planes=False, vel=vel)
    a, b = _pair(sc)
    errors = []
    for d in (a, b):
        d.step(3, 1)
        with pytest.raises(DemeError) as e:
            d.step(400, 1)
        errors.append(str(e.value))
    assert errors[0] == errors[1]
    assert a.counts().nSteps == b.counts().nSteps
    sa, sb = a.get_state(), b.get_state()
    for k in sa:
        assert np.array_equal(sa[k], sb[k]), k


@pytest.mark.parametrize("steps", [1, 9])
def test_lists_kept_over_replaced_states(steps):
    """States written between calls: moved a little (the lists hold), shuffled over the whole box (stale, again and again),
    back to an earlier one; the contact-list path builds anew each pass."""
    sc = scenes.sphere_settling(n=3001, spacing=1.98, velocity_sigma=0.3, seed=57)
    a, b = _pair(sc)
    rng = np.random.default_rng(4)
    where = ("voxelID", "locX", "locY", "locZ")
    first = None
    for k, move in enumerate(["jitter", "jitter", "shuffle", "shuffle", "shuffle", "first", "jitter", "shuffle", "jitter"]):
        for d in (a, b):
            d.step(steps)
        _same(a, b)
        st = a.get_state()
        first = first or {f: v.copy() for f, v in st.items()}
        if move == "jitter":
            st["locY"] ^= np.uint16(1 + k)
        elif move == "shuffle":
            p = np.arange(sc.n_owners)
            rng.shuffle(p[:sc.n_clumps])
            for f in where:
                st[f] = st[f][p]
        else:
            st = first
        for d in (a, b):
            d.set_state(st)
    for d in (a, b):
        d.step(steps)
    _same(a, b)


@pytest.mark.parametrize("how", ["ahead of time", "user model", "captured"])
def test_margin_lists_tested_first_equal_all_through_the_model(how):
    """A list of over 1M contacts with a drift margin, a sixth of them touching: tested in groups of 256 and packed,
    against every contact through the model (the cell sweep knows no share that touches). Calls end within and between
    detection passes; plane contacts' sums are folded from their places."""
    sc = scenes.clump_settling(n_clumps=100_003, update_freq=5, beta_frac=0.2, velocity_sigma=0.3, omega_sigma=5.0,
                               seed=58)
    a, b = _pair(sc, (lambda d: d.set_force_model(LINEAR, ["contact_age"])) if how == "user model" else None)
    if how == "captured":
        a.set_step_graphs(True)
    for chunk in (7, 3, 1, 14):
        a.step(chunk, 5)
        b.step(chunk, 5)
        _same(a, b)
    assert a.counts().nContacts > 1_000_000 and a.counts().nContacts % 256
    assert a.path_stats()[2] > 0 and b.path_stats()[2] == 0


def test_a_failed_list_build_leaves_no_lists():
    """A build that fails part-way (lists due for renewal, a sphere outside the world), then the state that the old lists
    were built from: the next call builds anew instead of stepping on lists that are half the old build's. The other
    system has its lists dropped by hand after the error."""
    r, skin, v, h = 0.005, 1e-3, 2.0, 1e-5
    g = np.stack(np.meshgrid(*[np.arange(6)] * 3, indexing="ij"), -1).reshape(-1, 3) * (2 * r * 0.9999)
    xyz = np.concatenate([g - g.mean(0), [[0.055, 0.055, -0.055]]])
    vel = np.random.default_rng(5).normal(0, 0.01, xyz.shape)
    vel[-1] = (0.0, 0.0, v)
    sc = scenes.spheres_scene(xyz, r, (0.1295, 0.1295, 0.1295), vel=vel, g=(0.0, 0.0, 0.0), planes=False, h=h)
    # single steps until a pass renews the lists ahead of time (before they are stale, at one skin of the lone sphere's
    # path: passes subtract the midpoint of the displacements): one step fewer leaves them due
    probe = DeviceSystem(sc)
    probe.set_skin(skin)
    n = 0
    while probe.candidate_stats()[2] < 2:
        probe.step(1)
        n += 1
    assert 4 < n and n * v * h < 0.95 * skin
    a, b = DeviceSystem(sc), DeviceSystem(sc)
    for d in (a, b):
        d.set_skin(skin)
        for _ in range(n - 1):
            d.step(1)
        assert d.candidate_stats()[2] == 1
        bad = d.get_state()
        z = np.uint64(sc.params.nvXp2 + sc.params.nvYp2)
        bad["voxelID"][-1] |= (~np.uint64(0) >> z) << z  # the last voxel in z: past the grid by its radius
        d.set_state(bad)
        with pytest.raises(DemeError):
            d.step(1)  # (too short for steps on the candidates, whose own check would end them)
        assert d.counts().nContacts > 200
        if d is b:
            d.set_skin(skin)
        d.set_state(sc.state)
        d.step(20)
    _same(a, b)


def test_margin_lists_destroy_histories_as_the_caller_says():
    """A long margin list whose non-touching contacts get a caller's history instead of zeros."""
    sc = scenes.clump_settling(n_clumps=100_003, update_freq=5, beta_frac=0.2, velocity_sigma=0.3, omega_sigma=5.0,
                               seed=58)
    away = "delta_tan_x = 0.f; delta_tan_y = 0.f; delta_tan_z = 0.f; delta_time -= 1.f;"
    a, b = _pair(sc, lambda d: d.jit_build({"_forceModelContactWildcardDestroy_": away}))
    for chunk in (7, 3, 6):
        a.step(chunk, 5)
        b.step(chunk, 5)
        _same(a, b)
    assert a.counts().nContacts > 1_000_000
    assert (a.wildcards()[3] <= -1.0).mean() > 0.5
    assert a.path_stats()[2] == 0


def _grazing_past_the_grid(m=17):
    """A bin grid one bin wide in x. A pair at its upper end in x grazes along y: the contact point, moved past the lower
    sphere's top by the rounding of the direction, falls into the next bin in y, which the sphere's linear bin ids hold
    only because its range in x passes the grid's end (bin (1, j) is bin (0, j + 1)). A cloud with many near neighbours
    makes a thinner skin pay at once."""
    f32 = np.float32
    r, rb, face = 0.005, 0.05, 0.5
    ra64, rb64 = np.float64(f32(r)), np.float64(f32(rb))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3) * (2.1 * r)
    xyz = np.concatenate([[[0.498, 0.49, 0.3], [0.498, 0.56, 0.3]], g + np.array([0.1, 0.6, 0.1])])
    rad = np.full(len(xyz), r)
    rad[1] = rb
    sc = scenes.spheres_scene(xyz - 0.5, rad, (1.0, 1.0, 1.0), lbf=(-0.5, -0.5, -0.5), planes=False, g=(0, 0, 0))
    p = sc.params
    p.binSize, p.nbX, p.nbY, p.nbZ = face, 1, 4, 4

    def enc(v):
        k = int(v // p.voxelSize)
        return k, int(round((v - k * p.voxelSize) / p.l))

    def dec(q):
        return np.float64(q[0]) * p.voxelSize + np.float64(q[1]) * p.l

    rng = np.random.default_rng(0)
    for _ in range(20000):
        t = rng.uniform(1e-4, 6e-4)
        qa = [enc(v) for v in (0.498, face - r - 8e-10, 0.3)]
        a = np.array([dec(q) for q in qa])
        d = ra64 + rb64 - 2e-10
        qb = [enc(v) for v in (a[0] + d * np.sin(t), a[1] + d * np.cos(t), a[2])]
        b = np.array([dec(q) for q in qb])
        if max(q[1] for q in qa + qb) > 65535 or ((a - b) ** 2).sum() > (ra64 + rb64) ** 2:
            continue
        n = (a - b).astype(f32)
        n /= np.sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2])
        half = (ra64 + rb64 - np.sqrt(((a - b) ** 2).sum())) / 2
        c = b + (rb64 - half) * n.astype(np.float64)
        if a[1] / face + ra64 / face < 1.0 <= c[1] / face:
            break
    else:
        raise AssertionError("no such pair")
    for k, q in enumerate((qa, qb)):
        sc.state["voxelID"][k] = q[0][0] | q[1][0] << p.nvXp2 | q[2][0] << (p.nvXp2 + p.nvYp2)
        for f, v in zip(("locX", "locY", "locZ"), q):
            sc.state[f][k] = v[1]
    return sc


def test_a_skin_narrowed_on_entry_keeps_the_check_of_the_state():
    """The state is checked against the grid's end although the call's first act is to rebuild its lists."""
    a, b = _pair(_grazing_past_the_grid())
    for chunk in (1, 1, 2000):
        for d in (a, b):
            d.step(chunk)
        assert chunk > 1 or b.counts().nContacts == 1
        _same(a, b)
    assert a.candidate_stats()[0] < 0.5 * b.scene.sph_radius.mean() * 0.2 and a.candidate_stats()[2] == 2
    assert a.path_stats()[:2] == (0, 1)  # narrowed on entry, and no step taken from that state


def test_a_calm_system_made_fast_gets_wider_lists():
    """Thin lists of a system at rest, then all spheres at 0.04 radii a step: the lists must come to last some steps."""
    r = 0.005
    g = np.stack(np.meshgrid(*[np.arange(17)] * 3, indexing="ij"), -1).reshape(-1, 3) * (2.1 * r)
    sc = scenes.spheres_scene(g - g.mean(0), r, (0.3, 0.3, 0.3), g=(0.0, 0.0, 0.0))
    a, b = _pair(sc)
    for d in (a, b):
        d.step(1)
        d.step(2000)
    assert a.candidate_stats()[0] < 0.05 * r
    v = np.random.default_rng(6).normal(size=(sc.n_clumps, 3))
    v *= 0.04 * r / sc.params.h / np.linalg.norm(v, axis=1, keepdims=True)
    st = a.get_state()
    for k, f in enumerate(("vX", "vY", "vZ")):
        st[f][:sc.n_clumps] = v[:, k]
    before = a.candidate_stats()[2]
    for d in (a, b):
        d.set_state(st)
        d.step(300)
    _same(a, b)
    assert a.candidate_stats()[0] > 0.25 * r
    assert a.candidate_stats()[2] - before < 300 / 4


def test_lists_that_never_last_give_way_to_the_cell_sweep():
    sc, _ = _fast_gas()
    a = DeviceSystem(sc)
    a.step(1)
    a.step(40)
    assert a.candidate_stats()[0] == 0.0
    builds = a.candidate_stats()[2]
    assert builds < 20
    a.step(200)
    assert a.candidate_stats()[2] < builds + 20


@pytest.mark.parametrize("how", ["free", "freed by a rule", "rule on its force"])
def test_a_plate_that_its_contacts_move_does_not_depend_on_the_lists(how):
    """A light plate thrown onto a bed: its accelerations move it, so their last bits must be those of the contact list
    whatever the lists and however the steps are split into calls. It is free from the start, or let go by a family
    change rule within a call, or held by a rule that reads its acceleration."""
    n = 1500
    sc = scenes.sphere_settling(n=n, spacing=1.98, jitter=0.0, velocity_sigma=0.2, omega_sigma=5.0, seed=61)
    top = float(scenes.decode_positions(sc.params, *(sc.state[k] for k in ("voxelID", "locX", "locY", "locZ")))[:n, 2].max())
    nc = sc.n_clumps
    extra = np.zeros(1, ANAL_DTYPE)
    extra[0]["owner"] = nc + 1
    extra[0]["relPos"] = (0.0, 0.0, top + 0.97 * 0.005)
    extra[0]["rot"] = (0.0, 0.0, -1.0)
    extra[0]["mass"] = 0.3
    sc.anal = np.concatenate([sc.anal, extra])
    sc.state = {q: np.concatenate([v, v[nc:nc + 1]]) for q, v in sc.state.items()}
    sc.state["family"][nc + 1] = 0 if how == "free" else 9
    sc.state["vZ"][nc + 1] = -0.2
    rule = np.zeros(1, RULE_DTYPE)[0]
    rule["used"] = rule["linVelPrescribed"] = rule["rotVelPrescribed"] = 1
    sc.rules[9] = rule
    sc.n_owners = nc + 2
    sc.owner_mass = np.append(sc.owner_mass, np.float32(0.3))
    sc.owner_moi = np.ascontiguousarray(np.append(sc.owner_moi, np.full((1, 3), 0.003, np.float32), 0))
    rules = {"free": None, "freed by a rule": "if (family_code == 9 && t > 2.35e-4f) newFamily = 0;",
             "rule on its force": "if (family_code == 9 && acc.z > 2.0f) newFamily = 0;"}[how]
    setup = (lambda d: d.set_motion_rules(family_change_rules=rules)) if rules else None
    a, b = _pair(sc, setup)
    c = DeviceSystem(sc)  # the automatic skin again, other calls
    if setup:
        setup(c)
    total = 0
    for chunk in (1, 40, 7, 60, 1, 90):
        for d in (a, b):
            d.step(chunk)
        total += chunk
        _same(a, b)
    for _ in range(total // 9):
        c.step(9)
    c.step(total % 9)
    sa, sb = a.get_state(), c.get_state()
    for k in sa:
        assert np.array_equal(sa[k], sb[k]), k
    assert sa["vZ"][nc + 1] != sc.state["vZ"][nc + 1] and sa["omgX"][nc + 1] != 0.0
    # the step that held the plate back, and those before it was let go
    assert a.path_stats()[0] >= (20 if how == "freed by a rule" else 1) and c.path_stats()[0] >= 1


def test_margin_lists_over_six_plane_owners():
    """Six floors of as many owners: the kernel that tests a long margin list first marks and folds each as the other kernel
    does."""
    sc = scenes.clump_settling(n_clumps=100_003, update_freq=5, beta_frac=0.2, velocity_sigma=0.3, omega_sigma=5.0,
                               seed=58)
    nc = sc.n_clumps
    sc.anal[:] = sc.anal[0]
    sc.anal["owner"] = nc + np.arange(len(sc.anal))
    sc.anal["relPos"][:, 2] += 1e-6 * np.arange(len(sc.anal), dtype=np.float32)
    more = len(sc.anal) - 1
    sc.state = {q: np.concatenate([v] + [v[nc:nc + 1]] * more) for q, v in sc.state.items()}
    sc.n_owners = nc + 1 + more
    sc.owner_mass = np.append(sc.owner_mass, np.full(more, 1e15, np.float32)).astype(np.float32)
    sc.owner_moi = np.ascontiguousarray(np.append(sc.owner_moi, np.full((more, 3), 1e15, np.float32), 0))
    a, b = _pair(sc)
    for chunk in (7, 3, 11):
        a.step(chunk, 5)
        b.step(chunk, 5)
        _same(a, b)
    assert a.counts().nContacts > 1_000_000
    assert np.all(a.get_state()["aZ"][nc:] != 0.0)
    assert a.path_stats()[2] > 0 and b.path_stats()[2] == 0


def test_a_list_that_outgrows_its_buffers_within_a_call():
    """A lattice without a contact closes up during one call: the contact list that the call ends in, and the one that a
    rebuild on the way hands its histories through, are many times longer than the buffers the call began with."""
    r = 0.005
    g = np.stack(np.meshgrid(*[np.arange(14)] * 3, indexing="ij"), -1).reshape(-1, 3) * (2.01 * r)
    g -= g.mean(0)
    sc = scenes.spheres_scene(g, r, (0.4, 0.4, 0.4), vel=-60.0 * g, g=(0.0, 0.0, 0.0), planes=False)
    a, b = _pair(sc)
    for chunk, least in ((1, 0), (30, 500), (20, 1000)):
        a.step(chunk)
        b.step(chunk)
        _same(a, b)
        assert a.counts().nContacts >= least and (chunk > 1 or a.counts().nContacts == 0)
    assert a.path_stats()[0] >= 40
