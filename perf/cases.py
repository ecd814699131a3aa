"""The work that users of this package have it do, one pass at a time.

A reconstruction program keeps the detector, the algorithm objects and the
uploaded events, calls an operator and reads its result.  Each case here is
one such call (or the two or three calls that always follow each other), on
simulated events of the package's own workloads (`simulation.workload`):

  find         the combinatorial Kalman filter on uploaded events, tracks read back
  progressive  the same with run_pkf: one branch per seed, no step structure
  prune        the filter with the learned branch scorer, tracks read back
  label        the filter that logs its branches, the scorer's training rows
               (features and labels stay on the GPU, where training reads them)
  fit          Kalman fit and smoother of an event's candidates, everything read back
  clean        fit of the candidates, then greedy ambiguity resolution of the
               fitted tracks, as the end of a reconstruction chain
  seed         spacepoints, triplet seeds and their track parameters of one event
  resolve      greedy ambiguity resolution of tracks already on the GPU
  train        the scorer from nothing: normalisation, training, logits of the rows

A program that takes event after event keeps the arrays that it reads results
into, as the C interface expects (include/traccc_amd/ckf.h, fitting.h,
seeding.h: buffers of the caller's).  The cases do the same: results go
through that interface into arrays with room for more, which `run` returns
with the number of entries that hold this pass's results.

`particles` is the number of particles of each event; with `least` the events
of a batch have between `least` and `particles`, evenly over the logarithm.
`tracks` and `rows` are the sizes of the last two kinds.
"""
import ctypes as C
import dataclasses
import math

import numpy as np
import torch

from traccc_amd import _ffi as F
from traccc_amd import ambiguity as AMB
from traccc_amd import ckf
from traccc_amd import fitting as FT
from traccc_amd import scorer as SC
from traccc_amd import seeding as SD
from traccc_amd import simulation as S

# simulation's own detectors and spectra: measurements a particle leaves (noise
# among them), measurements on one of its tracks, and how many more tracks a
# seed has with several branches per surface in an event of 60,000 particles
# (about in proportion to the event's size).
HITS = {"C1": 4.8, "C2": 5.8, "C3": 5.8, "C4": 6.0, "C5": 7.2}
ON_TRACK = {"C1": 4.4, "C2": 5.2, "C3": 5.2, "C4": 5.2, "C5": 6.1}
MORE = {"C1": 0.1, "C2": 1.0, "C3": 1.0, "C4": 3.0, "C5": 4.1}


def listed():
    return [
        # the smallest call: a test beam or an alignment event, a hundred muons in
        # a bare barrel; launches, read-backs and copies are all there is to it
        {"name": "find 100 muons", "call": "find", "workload": "C1", "events": 1, "particles": 100, "branches": 1},
        # one event by itself, as an online program gets them: barrel and disks
        # with material and noise, 10,000 muons
        {"name": "find 10k muons", "call": "find", "workload": "C2", "events": 1, "particles": 10000, "branches": 1},
        # offline reconstruction: events of very different sizes in one call, with
        # the field map in place of a constant field
        {"name": "find batch in map", "call": "find", "workload": "C3", "events": 8, "particles": 50000,
         "least": 500, "branches": 1},
        # the dense event: 60,000 pions, dead modules, noise, three branches per
        # surface, so most of the work is in branches that compete
        {"name": "find 60k pions", "call": "find", "workload": "C5", "events": 1, "particles": 60000, "branches": 3},
        # one branch per seed: the fast filter used where a trigger decides
        {"name": "progressive 10k muons", "call": "progressive", "workload": "C2", "events": 1, "particles": 10000,
         "branches": 1},
        # dense events with the scorer pruning branches: the package's headline path
        {"name": "prune 2x60k pions", "call": "prune", "workload": "C5", "events": 2, "particles": 60000, "branches": 3},
        # training rows for that scorer from the same kind of events
        {"name": "label 2x60k pions", "call": "label", "workload": "C5", "events": 2, "particles": 60000, "branches": 3},
        # precision analysis: every filtered and smoothed state of one event read back
        {"name": "fit 10k muons", "call": "fit", "workload": "C2", "events": 1, "particles": 10000, "branches": 1},
        # the end of the chain on dense events: fitted, then the ambiguous ones dropped
        {"name": "clean 2x60k pions", "call": "clean", "workload": "C5", "events": 2, "particles": 60000, "branches": 3},
        # seeding of one event, whose seeds the filter takes next
        {"name": "seed 10k muons", "call": "seed", "workload": "C2", "events": 1, "particles": 10000},
        # ambiguity resolution by itself, for tracks that another program found
        {"name": "resolve 1M tracks", "call": "resolve", "tracks": 1000000},
        # training on the rows of one event and more: 65,536 rows a step
        {"name": "train 2M rows", "call": "train", "rows": 2000000, "batch": 65536, "epochs": 3},
    ]


def draw(rng):
    """One more case of the same ranges: sizes over their logarithm, odd ones as they fall."""
    def size(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    call = rng.choice(["find", "find", "find", "progressive", "prune", "label", "fit", "clean", "seed", "resolve", "train"])
    if call == "resolve":
        return {"call": call, "tracks": size(1000, 1000000)}
    if call == "train":
        return {"call": call, "rows": size(50000, 2000000), "batch": rng.choice([16384, 65536]), "epochs": rng.choice([1, 2, 3])}
    if call == "seed":
        return {"call": call, "workload": rng.choice(["C2", "C4"]), "events": 1, "particles": size(100, 10000)}
    if call in ("prune", "label", "clean"):
        return {"call": call, "workload": rng.choice(["C4", "C5"]), "events": rng.choice([1, 2]),
                "particles": size(1000, 60000), "branches": 3}
    if call == "fit":
        return {"call": call, "workload": rng.choice(["C2", "C3", "C4"]), "events": 1, "particles": size(100, 10000), "branches": 1}
    if call == "progressive":
        return {"call": call, "workload": rng.choice(["C2", "C3", "C4"]), "events": 1, "particles": size(100, 20000), "branches": 1}
    workload = rng.choice(["C1", "C2", "C3", "C4", "C5"])
    case = {"call": call, "workload": workload, "events": rng.choice([1, 1, 2, 3, 5, 8]), "particles": size(50, 10000),
            "branches": rng.choice([1, 1, 2, 3])}
    if case["events"] > 1 and rng.random() < 0.5:
        case["least"] = max(20, case["particles"] // 100)
    return case


def counts(case):
    """Particles of each event: one number, or spread over the logarithm from `least`."""
    n = case["events"]
    if not case.get("least"):
        return [case["particles"]] * n
    a, b = math.log(case["least"]), math.log(case["particles"])
    return [int(round(math.exp(a + (b - a) * (k + 0.5) / n))) for k in range(n)]


def simulated(case, seed):
    """Detector, field and events; the sizes of a batch come in an order of the seed's."""
    det, fld, gun = S.workload(case["workload"], seed=seed)
    sizes = counts(case)
    np.random.default_rng(seed).shuffle(sizes)
    guns = [dataclasses.replace(gun, n_particles=n, seed=1000003 * (seed % 1000000) + e) for e, n in enumerate(sizes)]
    return det, fld, S.generate_events(det, fld, guns)


def pruning_scorer(seed):
    """A scorer that weighs candidates as trained ones do: chi2, the running
    chi2 / ndf, the standing among the seed's branches and the rank count
    against a candidate.  GELU(x) - GELU(-x) = x, so pairs of hidden units
    carry the sum through both layers; the other units are a trained net's
    leftovers, small and random."""
    r = np.random.default_rng(seed)
    w1 = r.normal(0.0, 0.02, (12, 64))
    w2 = r.normal(0.0, 0.02, (64, 64))
    w3 = r.normal(0.0, 0.02, 64)
    mean = np.array([0, 0, 2.5, 0.5, 0, 1.57, 0.2, 4.0, 1.2, 0.6, 0.4, 0.9], np.float32)
    std = np.array([1, 1, 3.5, 0.3, 1, 0.9, 0.5, 3.0, 1.0, 1.2, 0.6, 0.4], np.float32)
    weight = {2: -1.6, 8: -0.4, 9: -1.5, 10: -0.8, 7: 0.2}
    w1[:, :2], w2[:2, :2], w3[:2] = 0.0, 0.0, 0.0
    for f, w in weight.items():
        w1[f, 0], w1[f, 1] = w, -w
    w2[0, 0] = w2[1, 1] = 1.0
    w2[1, 0] = w2[0, 1] = -1.0
    w3[0], w3[1] = 1.0, -1.0
    params = np.concatenate([w1.reshape(-1), np.zeros(64), w2.reshape(-1), np.zeros(64), w3, [0.5]])
    scorer = SC.Scorer(seed=seed)
    scorer.set_params(params.astype(np.float32), mean, std)
    return scorer


def training_rows(n, seed):
    """Branch rows as the filter logs them (scorer.FEATURE_NAMES) and labels that follow them."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def normal():
        return torch.randn(n, device="cuda", generator=g)

    def uniform():
        return torch.rand(n, device="cuda", generator=g).clamp_(1e-6, 1 - 1e-6)

    pull0, pull1 = 1.1 * normal(), 1.1 * normal()
    chi2 = (pull0 * pull0 + pull1 * pull1).clamp_(max=30.0)
    depth = torch.floor(9.0 * uniform())
    running = -torch.log(uniform())
    standing = torch.relu(-1.5 * torch.log(uniform()) - 1.2)
    rank = torch.floor(3.0 * uniform() ** 2)
    x = torch.stack([pull0, pull1, chi2, uniform(), normal(), 3.1 * uniform(), torch.floor(1.3 * uniform()), depth,
                     running, standing, rank, torch.log1p(rank + torch.floor(1.0 + 4.0 * uniform()))], dim=1)
    logit = 1.0 - 0.45 * (chi2 - 2.4) - 1.2 * standing - 0.7 * rank - 0.3 * running
    labels = (uniform() < torch.sigmoid(logit)).to(torch.uint8)
    return x.contiguous(), labels


def synthetic_tracks(n, seed):
    """Track candidates as a dense event gives them: each particle is found a
    few times, the copies share most of its measurements, some hold a
    neighbour's.  Events of up to 30,000 particles one after another, tracks
    ordered by their length in each, measurement identifiers by layer."""
    r = np.random.default_rng(seed)
    layers = 9
    copies = r.choice([1, 2, 3, 4, 6, 9], size=n, p=[0.45, 0.2, 0.12, 0.1, 0.08, 0.05])
    particle = np.repeat(np.arange(n), copies)[:n]
    n_part = int(particle[-1]) + 1
    n_ev = -(-n_part // 30000)
    per = -(-n_part // n_ev)
    event = particle // per
    length = np.clip(r.integers(4, layers + 1, n_part)[particle] - (r.random(n) < 0.3), 3, layers)
    hit = np.arange(layers)[None, :] < length[:, None]
    at = np.where(r.random((n, layers)) < 0.07, r.integers(0, per, (n, layers)), (particle % per)[:, None])
    place = np.stack([r.permutation(per) for _ in range(layers)])
    ids = (event[:, None] * layers + np.arange(layers)[None, :]) * per + place[np.arange(layers)[None, :], at]
    order = np.lexsort((particle, length, event))
    hit, ids, length = hit[order], ids[order], length[order]
    offsets = np.concatenate([[0], np.cumsum(length)]).astype(np.int32)
    pvals = r.random(n).astype(np.float32)
    return (torch.from_numpy(offsets).cuda(), torch.from_numpy(ids[hit].astype(np.int32)).cuda(),
            torch.from_numpy(pvals).cuda(), int(n_ev * layers * per))


def finding_config(case):
    cfg = S.finding_config_for(case["workload"])
    cfg.max_num_branches_per_surface = case["branches"]
    cfg.run_pkf = int(case["call"] == "progressive")
    return cfg


def arrays(tracks, entries, kinds):
    """Arrays of the program's own for `tracks` tracks with `entries` entries in
    all, by name: kinds gives (type, width, which of the two counts)."""
    made = {}
    for name, (dtype, width, count) in kinds.items():
        n = {"tracks": tracks, "ends": tracks + 1, "entries": entries}[count]
        made[name] = np.full((n, width) if width > 1 else n, 0, dtype)
    return made


TRACK = {"fit_outcome": (np.uint16, 1, "tracks"), "params_surface_link": (np.uint64, 1, "tracks"),
         "params_vector": (np.float32, 6, "tracks"), "params_covariance": (np.float32, 36, "tracks"),
         "ndf": (np.float32, 1, "tracks"), "chi2": (np.float32, 1, "tracks"), "pval": (np.float32, 1, "tracks"),
         "nholes": (np.uint32, 1, "tracks")}
CANDIDATES = {**TRACK, "constituent_offsets": (np.uint32, 1, "ends"), "constituent_type": (np.uint16, 1, "entries"),
              "constituent_index": (np.uint32, 1, "entries")}
FITTED = {**TRACK, "state_offsets": (np.uint32, 1, "ends"), "state_flags": (np.uint8, 1, "entries"),
          "filtered_chi2": (np.float32, 1, "entries"), "smoothed_chi2": (np.float32, 1, "entries"),
          "backward_chi2": (np.float32, 1, "entries"), "state_surface_link": (np.uint64, 1, "entries"),
          "filtered_vector": (np.float32, 6, "entries"), "filtered_covariance": (np.float32, 36, "entries"),
          "smoothed_vector": (np.float32, 6, "entries"), "smoothed_covariance": (np.float32, 36, "entries"),
          "measurement_index": (np.uint32, 1, "entries")}


def bind(struct, made):
    """The interface's struct over those arrays."""
    for name, column in made.items():
        setattr(struct, name, column.ctypes.data_as(type(getattr(struct, name))))
    return struct


def checked(status):
    if status != 0:
        raise RuntimeError(F.load_library(ckf.LIB).ckf_last_error().decode())


def found(case, particles):
    """Tracks found for each seed in an event of that many particles."""
    if case["branches"] == 1:
        return 1.0
    more = MORE[case["workload"]] * (particles / 60000.0) ** 1.1
    return 1.0 + (0.05 if case["call"] == "prune" else 1.0) * more


def room(case, seeds):
    """Tracks and measurements on them that the program's arrays hold."""
    most = found(case, max(counts(case)))
    tracks = int((1.5 * most + (0.0 if case["branches"] == 1 else 0.6)) * seeds) + 500
    return tracks, int(1.6 * HITS[case["workload"]] * tracks)


def prepare(case, seed):
    call = case["call"]
    s = {"call": call}
    if call == "resolve":
        s["resolver"] = AMB.greedy_ambiguity_resolution_algorithm()
        s["tracks"] = synthetic_tracks(case["tracks"], seed)
        return s
    if call == "train":
        s["rows"], s["labels"] = training_rows(case["rows"], seed)
        s["config"] = SC.train_config(epochs=case["epochs"], batch=case["batch"],
                                      learning_rate=4e-3 if case["batch"] > 16384 else 2e-3)
        return s
    det, fld, events = simulated(case, seed)
    s["detector"] = ckf.DeviceDetector(det, fld)
    s["events"] = ckf.DeviceEvents(s["detector"], events)
    if call == "seed":
        finder = SD.seedfinder_config(bFieldInZ=2.0 * SD.TESLA)
        s["seeder"] = SD.seeding_algorithm(finder, SD.spacepoint_grid_config(finder), SD.seedfilter_config())
        s["estimation"] = SD.track_params_estimation_config()
        s["measurements"] = events[0].measurements_struct()
        s["event"] = events[0]
        s["field"] = (C.c_float * 3)(0.0, 0.0, 2.0 * SD.TESLA)
        points, seeds = int(1.3 * HITS[case["workload"]] * case["particles"]) + 500, 40 * case["particles"] + 2000
        s["points"] = {"xyz": np.full((points, 3), 0, np.float32), "index": np.full(points, 0, np.uint32)}
        s["seeds"] = {"bottom": np.full(seeds, 0, np.uint32), "middle": np.full(seeds, 0, np.uint32),
                      "top": np.full(seeds, 0, np.uint32), "weight": np.full(seeds, 0, np.float32)}
        s["parameters"] = {"surface": np.full(seeds, 0, np.uint64), "vector": np.full((seeds, 6), 0, np.float32),
                           "covariance": np.full((seeds, 36), 0, np.float32)}
        return s
    cfg = finding_config(case)
    s["finder"] = ckf.combinatorial_kalman_filter_algorithm(cfg)
    n_tracks, n_entries = room(case, s["events"].n_seeds)
    if call == "label":
        rows = 26 * s["events"].n_seeds
        s["rows"] = torch.zeros((rows, SC.N_FEATURES), dtype=torch.float32, device="cuda")
        s["labels"] = torch.zeros(rows, dtype=torch.uint8, device="cuda")
        return s
    if call in ("fit", "clean"):
        s["candidates"] = s["finder"].run_device(s["detector"], s["events"])
        del s["finder"]
        s["fitter"] = FT.kalman_fitting_algorithm(FT.fitting_config(cfg))
        if call == "fit":
            s["out"] = arrays(n_tracks, n_entries, FITTED)
        else:
            s["resolver"] = AMB.greedy_ambiguity_resolution_algorithm()
            s["keep"] = np.full(n_tracks, 0, np.uint8)
        return s
    if call == "prune":
        s["scorer"] = pruning_scorer(seed)
        s["finder"].set_scorer(s["scorer"], threshold=-1.5)
    s["out"] = arrays(n_tracks, n_entries, CANDIDATES)
    return s


def read_back(result, out, struct, download):
    """A result's sizes and, in the program's arrays, its columns."""
    n, entries = result.sizes()
    if n + 1 > len(next(v for k, v in out.items() if k.endswith("_offsets"))) or entries > len(list(out.values())[-1]):
        raise RuntimeError("%d tracks, %d entries: more than the arrays hold" % (n, entries))
    struct = bind(struct, out)
    struct.n_tracks, checks = n, entries
    if hasattr(struct, "n_states"):
        struct.n_states = checks
    checked(download(result._h, C.byref(struct)))
    return {"n": n, "entries": entries, **out}


def find_seeds(s):
    """Spacepoints, seeds and their parameters, one call of the interface after the other."""
    lib = SD._lib()
    points, seeds, made = s["points"], s["seeds"], s["parameters"]
    n = C.c_uint32()
    checked(lib.ckf_spacepoint_formation(s["detector"]._h, s["events"]._h, 0, None, None, C.byref(n)))
    n_points = n.value
    if n_points > len(points["index"]):
        raise RuntimeError("%d spacepoints: more than the arrays hold" % n_points)
    checked(lib.ckf_spacepoint_formation(s["detector"]._h, s["events"]._h, 0, points["xyz"].ctypes.data,
                                         points["index"].ctypes.data, C.byref(n)))
    sp = SD.Spacepoints(n_points, points["xyz"].ctypes.data, None, None, points["index"].ctypes.data)
    checked(lib.ckf_seeding_run(s["seeder"]._h, C.byref(sp), C.byref(n)))
    n_seeds = n.value
    if n_seeds > len(seeds["bottom"]):
        raise RuntimeError("%d seeds: more than the arrays hold" % n_seeds)
    struct = SD.Seeds(n_seeds, *[v.ctypes.data for v in seeds.values()])
    checked(lib.ckf_seeding_result_download(s["seeder"]._h, C.byref(struct)))
    checked(lib.ckf_estimate_track_params(C.byref(s["estimation"]), C.byref(sp), C.byref(struct),
                                          C.byref(s["measurements"]), C.byref(s["field"]),
                                          *[v.ctypes.data for v in made.values()]))
    return {"n_points": n_points, "n_seeds": n_seeds, **points, **seeds, **made}


def run(s):
    call = s["call"]
    if call in ("find", "progressive", "prune"):
        tracks = s["finder"].run_device(s["detector"], s["events"])
        return read_back(tracks, s["out"], F.TrackCandidates(), ckf._lib().ckf_tracks_download)
    if call == "label":
        n, tracks = C.c_uint32(), C.c_void_p()
        checked(ckf._lib().ckf_find_tracks_logged(s["finder"]._h, s["detector"]._h, s["events"]._h, s["rows"].data_ptr(),
                                                  s["labels"].data_ptr(), len(s["labels"]), C.byref(n), C.byref(tracks)))
        return {"n": n.value, "rows": s["rows"], "labels": s["labels"], "events": ckf.DeviceTracks(tracks).event_offsets()}
    if call == "fit":
        fitted = s["fitter"].run_device(s["detector"], s["events"], s["candidates"])
        return read_back(fitted, s["out"], F.FittedTracks(), FT._lib().ckf_fitted_download)
    if call == "clean":
        fitted = s["fitter"].run_device(s["detector"], s["events"], s["candidates"])
        n, _ = fitted.sizes()
        if n > len(s["keep"]):
            raise RuntimeError("%d tracks: more than the array holds" % n)
        kept = C.c_uint32()
        checked(AMB._lib().ckf_resolve_fitted(s["resolver"]._h, s["events"]._h, fitted._h,
                                              s["keep"].ctypes.data_as(F.c_u8_p), C.byref(kept)))
        return {"n": n, "kept": kept.value, "keep": s["keep"]}
    if call == "seed":
        return find_seeds(s)
    if call == "resolve":
        offsets, ids, pvals, bound = s["tracks"]
        keep, kept = s["resolver"].run_device(offsets, ids, pvals, bound)
        return {"keep": keep, "kept": kept}
    scorer = SC.Scorer(seed=7)
    scorer.fit_normalisation(s["rows"])
    stats = scorer.train(s["rows"], s["labels"], s["config"])
    params, mean, std = scorer.params()
    return {"logits": scorer.forward(s["rows"]), "params": params, "mean": mean, "std": std,
            "losses": [stats.first_loss, stats.last_loss]}


def work(case):
    """Bytes: measurements 20 B, seeds 192 B, a track 200 B and 6 B a
    measurement of it, a fitted state 360 B, a row 48 B.  Operations: 4,000 for
    a branch over one surface (five Runge-Kutta steps with their derivatives,
    the covariance's transport, an update), half of that again to smooth it."""
    call = case["call"]
    if call == "resolve":
        n = case["tracks"]
        return {"bytes": n * (4 + 4 + 1 + 4 * 6.3), "flops": 0}
    if call == "train":
        n = case["rows"]
        mlp = 2.0 * (12 * 64 + 64 * 64 + 64)
        return {"bytes": n * (48 + 1 + 4), "flops": n * mlp * (3 * case["epochs"] + 1)}
    n = float(sum(counts(case)))
    hits = HITS[case["workload"]]
    if call == "seed":
        return {"bytes": n * hits * (20 + 16 + 16 + 176), "flops": n * hits * 500}
    sizes = counts(case)
    tracks = sum(m * found(case, m) for m in sizes)
    on_track = ON_TRACK[case["workload"]]
    # a seed's branches part along the way: a further track has most of its surfaces of its own
    steps = on_track * n + 0.75 * on_track * (tracks - n)
    read = n * (hits * 20 + 192)
    written = tracks * (200 + 6 * on_track)
    if call == "label":
        return {"bytes": read + steps * 49, "flops": steps * 4000}
    if call == "fit":
        return {"bytes": read + written + tracks * on_track * 360, "flops": tracks * on_track * 6000}
    if call == "clean":
        return {"bytes": read + tracks * 201, "flops": tracks * on_track * 6000}
    return {"bytes": read + written, "flops": steps * 4000}


def tolerance(case):
    """About four times what two correct builds in single precision differ by,
    measured with this package's CPU checker in 32 bits against the GPU.

    Positions along a track come from direction cosines over up to a metre of
    path (a 6e-8 error there is 1e-3 of a 50 um resolution), and chi2 terms are
    squares of residuals: chi2 5e-4 and p-values 8e-4 apart, 0.013 at most in
    one of them.  A whole value differs where two candidates' chi2 are that
    close.  The fit's filtered chi2 are 4e-3 apart, 0.04 at most.  Training:
    rows moved by 3e-7 of themselves move the logits by 4e-4, 0.008 at most.
    """
    call = case["call"]
    if call in ("find", "progressive", "prune", "label"):
        return {"rel": 3e-3, "max": 0.05, "differ": 1e-3}
    if call == "fit":
        return {"rel": 0.015, "max": 0.16, "differ": 1e-3}
    if call == "clean":
        return {"rel": 0.0, "differ": 1e-3}
    if call == "seed":
        return {"rel": 1e-5, "max": 1e-3, "differ": 0.0}
    if call == "resolve":
        return "exact"
    return {"rel": 2e-3, "max": 0.04}


def exact(case, seed):
    """In 64 bits: the spacepoints of an event from its surfaces, the
    normalisation of training rows.  The filter and the fit would be a second
    track finder here, and a training's 64-bit weights are other weights."""
    call = case["call"]
    if call == "seed":
        det, _, events = simulated(case, seed)
        ev = events[0]
        place = {int(det.surface(i).identifier): i for i in range(det.n_surfaces)}
        frame = np.array([[det.surface(i).center[:], det.surface(i).axis_u[:], det.surface(i).axis_v[:]]
                          for i in range(det.n_surfaces)], np.float64)
        pixel = ev.dimensions == 2
        at = np.array([place[int(v)] for v in ev.surface_link[pixel]])
        loc = ev.local_position[pixel].astype(np.float64)
        xyz = frame[at, 0] + loc[:, :1] * frame[at, 1] + loc[:, 1:] * frame[at, 2]
        points = np.zeros((int(1.3 * HITS[case["workload"]] * case["particles"]) + 500, 3))
        points[:len(xyz)] = xyz
        return {"n_points": len(xyz), "n_seeds": None, "xyz": points, "index": None, "bottom": None, "middle": None,
                "top": None, "weight": None, "surface": None, "vector": None, "covariance": None}
    if call == "train":
        x = training_rows(case["rows"], seed)[0].double()
        return {"logits": None, "params": None, "mean": x.mean(dim=0), "std": x.std(dim=0, unbiased=False), "losses": None}
    return None
