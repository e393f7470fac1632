"""Performance cases of the PPO learning path on one GPU: what a training
program has this library do, through its Python API.

The kinds of work, each over the range of sizes a user runs:

act      one rollout step: normalise the observations, actor, sampling,
         log-probabilities, critic values. From a handful of environments
         (launch latency counts) to tens of thousands.
returns  the end of a rollout: critic values of every sample and of the
         bootstrap observations, GAE, advantage normalisation.
layers   two feature-major layers through the GEMM adapter, forward and (with
         train) backward: gemm_bias_act, gemm, elu_backward, row_sum as the
         reference trainer's network calls them.
loss     the PPO loss gradients of a minibatch, actor and critic.
adam     the clipped Adam step over the tensors of an actor and a critic.
norm     the observation normaliser over a batch: push, commit, normalize.
grads    the gradients of one minibatch, both networks.
update   a whole PPO update, epochs x minibatches, then the parameters read
         back (a trainer publishes or saves them).

All arithmetic is fp32. Inputs are drawn on the GPU from the seed; the float64
results of exact() are plain torch on those inputs.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from zealot_amd import Context, DeviceBuffer, _ffi, ops
from zealot_amd.rl import GpuActorCritic, GpuNormalizer, GpuPendingNorm, PpoConfig

# The repository's networks: the headline pair, the reference trainer's pair
# (separate critic observation), a small generic pair with odd widths.
HEADLINE = ("123-512-256-128-29", "123-512-256-128-1")
TRAINER = ("265-256-256-128-12", "64-512-256-128-1")
SMALL = ("37-64-48-7", "37-64-48-1")

LOG_SQRT_2PI = 0.9189385
CLIP, ENTROPY, VALUE_COEF = 0.2, 0.005, 1.0
GAMMA, LAM = 0.99, 0.95
BETA1, BETA2, EPS = 0.9, 0.999, 1e-8
LOG_STD = -0.5


def listed():
    a, c = HEADLINE
    ta, tc = TRAINER
    return [
        # A debugging or evaluation run: few environments, latency only.
        {"name": "act_64", "kind": "act", "actor": a, "critic": c, "envs": 64},
        # The rollout step of the headline workload.
        {"name": "act_4096", "kind": "act", "actor": a, "critic": c, "envs": 4096},
        # A large rollout on the reference trainer's networks, an odd number of rows.
        {"name": "act_20011", "kind": "act", "actor": ta, "critic": tc, "envs": 20011},
        # The end of the headline rollout (rows padded to 16 bytes by the caller).
        {"name": "returns_4096x24", "kind": "returns", "actor": a, "critic": c, "envs": 4096, "steps": 24, "pad": 4},
        # A single dense layer and its output, inference: the 123-wide input layer.
        {"name": "layers_fwd_4096", "kind": "layers", "in": 123, "mid": 512, "out": 29, "rows": 4096, "train": False},
        # The same through two wide layers of a minibatch, forward and backward.
        {"name": "layers_train_24576", "kind": "layers", "in": 512, "mid": 256, "out": 128, "rows": 24576, "train": True},
        # The loss gradients of a minibatch, the trainer's feature-major tensors.
        {"name": "loss_24576", "kind": "loss", "rows": 24576, "actions": 29, "feature_major": True},
        # The optimiser step over both headline networks.
        {"name": "adam_headline", "kind": "adam", "actor": a, "critic": c, "max_norm": 1.0},
        # The normaliser over the headline rollout.
        {"name": "norm_98304", "kind": "norm", "dim": 123, "rows": 98304, "pad": 1},
        # The gradients of one headline minibatch, read back.
        {"name": "grads_24576", "kind": "grads", "actor": a, "critic": c, "rows": 24576, "feature_major": False},
        # A small training run under ActorCritic::update: shuffled minibatches.
        {"name": "update_64x24", "kind": "update", "actor": a, "critic": c, "envs": 64, "steps": 24,
         "epochs": 5, "minibatches": 4, "trainer": False, "feature_major": False},
        # The headline update.
        {"name": "update_4096x24", "kind": "update", "actor": a, "critic": c, "envs": 4096, "steps": 24,
         "epochs": 5, "minibatches": 4, "trainer": True, "feature_major": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["act", "act", "returns", "layers", "layers", "loss", "adam", "norm", "grads", "grads",
                       "update", "update"])
    actor, critic = rng.choice([HEADLINE, HEADLINE, TRAINER, TRAINER, SMALL])
    fm = rng.random() < 0.5
    if kind == "act":
        return {"kind": kind, "actor": actor, "critic": critic, "envs": _log_int(rng, 8, 32768)}
    if kind == "returns":
        return {"kind": kind, "actor": actor, "critic": critic, "envs": _log_int(rng, 16, 4096),
                "steps": rng.randint(8, 24), "pad": rng.choice([1, 4])}
    if kind == "layers":
        return {"kind": kind, "in": _log_int(rng, 24, 512), "mid": rng.choice([64, 100, 128, 256, 512]),
                "out": rng.choice([12, 29, 64, 128, 256]), "rows": _log_int(rng, 512, 24576),
                "train": rng.random() < 0.6}
    if kind == "loss":
        return {"kind": kind, "rows": _log_int(rng, 256, 65536), "actions": rng.choice([6, 12, 29, 32, 40]),
                "feature_major": fm}
    if kind == "adam":
        return {"kind": kind, "actor": actor, "critic": critic, "max_norm": rng.choice([0.5, 1.0, 2.0]) + rng.randint(0, 99) / 100}
    if kind == "norm":
        return {"kind": kind, "dim": rng.choice([37, 45, 64, 123, 128, 265]), "rows": _log_int(rng, 256, 98304),
                "pad": rng.choice([1, 4])}
    if kind == "grads":
        return {"kind": kind, "actor": actor, "critic": critic, "rows": _log_int(rng, 256, 24576), "feature_major": fm}
    return {"kind": kind, "actor": actor, "critic": critic, "envs": _log_int(rng, 16, 4096), "steps": rng.randint(8, 24),
            "epochs": rng.randint(2, 5), "minibatches": rng.choice([2, 4, 5]), "trainer": rng.random() < 0.6,
            "feature_major": fm}


# ------------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _dims(text):
    return [int(x) for x in text.split("-")]


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _uniform(g, bound, *shape):
    return (torch.rand(*shape, generator=g, device="cuda") * 2 - 1) * bound


def _net(g, dims):
    """[(w [out x in], b [out])] per layer: Kaiming-uniform weights, small biases."""
    return [(_uniform(g, math.sqrt(6.0 / dims[i]), dims[i + 1], dims[i]), _uniform(g, 0.1, dims[i + 1]))
            for i in range(len(dims) - 1)]


def _packed(net):
    return torch.cat([t.reshape(-1) for w, b in net for t in (w, b)]).cpu().numpy()


def _forward(net, x):
    """Activations of every layer, x first, in the precision of the arguments."""
    acts = [x]
    for i, (w, b) in enumerate(net):
        z = acts[-1] @ w.t() + b
        acts.append(torch.where(z > 0, z, torch.expm1(torch.clamp(z, max=0.0))) if i + 1 < len(net) else z)
    return acts


def _double(net):
    return [(w.double(), b.double()) for w, b in net]


def _obs(g, rows, dim):
    return torch.clamp(_normal(g, rows, dim), -5.0, 5.0)


def _logp(action, mean, log_std):
    d = (action - mean) / torch.exp(log_std)
    return (-0.5 * d * d - log_std - LOG_SQRT_2PI).sum(1)


def _rollout(g, actor, critic, obs, cobs, A):
    """Actions, old log-probabilities and values, advantages and returns of
    rows that the policy itself produced a moment (one small update) ago.
    The losses are discontinuous: where a row's ratio lies on the clip
    boundary or its two value losses tie, the last bit of a sum decides its
    whole gradient, so such rows are moved off."""
    n = obs.shape[0]
    mean = torch.cat([_forward(_double(actor), x.double())[-1] for x in obs.split(32768)])
    v = torch.cat([_forward(_double(critic), x.double())[-1] for x in cobs.split(32768)])[:, 0]
    ls = torch.full((A,), LOG_STD, device="cuda")
    action = (mean + math.exp(LOG_STD) * _normal(g, n, A).double()).float()
    lp = _logp(action.double(), mean, ls.double())
    shift = 0.05 * _normal(g, n).double()
    for edge in (math.log(1 - CLIP), math.log(1 + CLIP)):
        shift = torch.where((shift - edge).abs() < 0.01, shift + 0.03, shift)
    logp_old = (lp - shift).float()
    mean_old = (mean + 0.02 * _normal(g, n, A).double()).float()
    value_old, ret = _value_targets(g, v)
    adv = _normal(g, n)
    return dict(action=action, mean_old=mean_old, logp_old=logp_old, value_old=value_old, adv=adv, ret=ret, log_std=ls)


def _value_targets(g, v):
    vo = v + 0.15 * _normal(g, v.shape[0]).double()
    ret = v + _normal(g, v.shape[0]).double()
    dv = v - vo
    vc = vo + torch.clamp(dv, -CLIP, CLIP)
    tie = ((v - ret) ** 2 - (vc - ret) ** 2).abs() < 1e-3
    near = (dv.abs() - CLIP).abs() < 1e-2
    vo = torch.where((near | (tie & (dv.abs() > CLIP))), v + 0.05, vo)
    return vo.float(), ret.float()


# ------------------------------------------------- the library's buffers

_context = None


def _ctx():
    global _context
    if _context is None:
        _context = Context(torch.cuda.current_device())
    return _context


class Buf(DeviceBuffer):
    """A torch tensor's memory as a DeviceBuffer (torch owns it)."""

    def __init__(self, tensor):
        self.tensor = tensor
        dtype = {torch.float32: np.float32, torch.uint8: np.uint8, torch.int32: np.int32}[tensor.dtype]
        super().__init__(_ctx(), tensor.data_ptr(), tensor.numel() * tensor.element_size(), tensor.shape, dtype)

    def free(self):
        self.ptr = 0


def _new(*shape):
    return Buf(torch.zeros(*shape, device="cuda"))


def _rows(x, pad):
    """Row-major rows of x with a stride rounded up to `pad` floats: (buffer, stride)."""
    n, d = x.shape
    ld = -(-d // pad) * pad
    y = torch.zeros(n, ld, device="cuda")
    y[:, :d] = x
    return Buf(y), ld


class Batch:
    """The batch of an update, as GpuActorCritic takes it."""

    def __init__(self, d, fm):
        f = (lambda x: x.t().contiguous()) if fm else (lambda x: x.contiguous())
        self.n = d["obs"].shape[0]
        self.fm = fm
        self.t = {k: f(d[k]) for k in ("obs", "action", "mean_old")}
        self.t["cobs"] = self.t["obs"] if d["cobs"] is d["obs"] else f(d["cobs"])
        # The update normalises adv in place: the copy is the rollout's own.
        self.t.update({k: d[k].clone() for k in ("logp_old", "value_old", "adv", "ret")})
        self.dims = (d["obs"].shape[1], d["cobs"].shape[1], d["action"].shape[1])

    def to_c(self):
        od, cd, A = self.dims
        ld = (lambda k: self.n) if self.fm else (lambda k: k)
        p = {k: x.data_ptr() for k, x in self.t.items()}
        bits = (_ffi.ZL_FM_OBS | _ffi.ZL_FM_CRITIC_OBS | _ffi.ZL_FM_ACTION | _ffi.ZL_FM_MEAN_OLD) if self.fm else 0
        return _ffi.zl_batch(self.n, p["obs"], ld(od), p["cobs"], ld(cd), p["action"], ld(A), p["mean_old"], ld(A),
                             p["logp_old"], p["value_old"], p["adv"], p["ret"], bits)


def _inputs(case, seed):
    """What the case computes on, as torch tensors (float32, on the GPU)."""
    g = _gen(seed)
    kind = case["kind"]
    d = {}
    if kind in ("act", "returns", "grads", "update", "adam"):
        ad, cd = _dims(case["actor"]), _dims(case["critic"])
        d.update(ad=ad, cd=cd, actor=_net(g, ad), critic=_net(g, cd))
    if kind == "act":
        n = case["envs"]
        for key, dim in (("obs", ad[0]), ("cobs", cd[0])):
            d[key] = _normal(g, n, dim) * 2 + 0.5
            mean, var, count = 0.5 + 0.1 * _normal(g, dim), 4 * (0.5 + torch.rand(dim, generator=g, device="cuda")), 50000.0
            d[key + "_state"] = torch.cat([mean, var * count, torch.tensor([count], device="cuda")])
        d["eps"] = _normal(g, n, ad[-1])
    elif kind == "returns":
        T, N = case["steps"], case["envs"]
        d["obs"], d["boot"] = _obs(g, T * N, cd[0]), _obs(g, N, cd[0])
        d["rewards"] = _normal(g, T, N)
        d["dones"] = (torch.rand(T, N, generator=g, device="cuda") < 0.02).to(torch.uint8)
    elif kind == "layers":
        i, m, o, n = case["in"], case["mid"], case["out"], case["rows"]
        d.update(x=_normal(g, i, n), w1=_uniform(g, math.sqrt(6.0 / i), m, i), b1=_uniform(g, 0.1, m),
                 w2=_uniform(g, math.sqrt(6.0 / m), o, m), b2=_uniform(g, 0.1, o), g2=_normal(g, o, n) / n)
    elif kind == "loss":
        n, A = case["rows"], case["actions"]
        mean = _normal(g, n, A)
        ls = LOG_STD + 0.2 * _normal(g, A)
        action = mean + torch.exp(ls) * _normal(g, n, A)
        lp = _logp(action.double(), mean.double(), ls.double())
        shift = 0.1 * _normal(g, n).double()
        for edge in (math.log(1 - CLIP), math.log(1 + CLIP)):
            shift = torch.where((shift - edge).abs() < 0.01, shift + 0.03, shift)
        v = _normal(g, n)
        vo, ret = _value_targets(g, v.double())
        d.update(mean=mean, action=action, log_std=ls, adv=_normal(g, n), logp_old=(lp - shift).float(),
                 mean_old=mean + 0.02 * _normal(g, n, A), v=v, value_old=vo, ret=ret)
    elif kind == "adam":
        d["p"] = [t for net in (d["actor"], d["critic"]) for w, b in net for t in (w.reshape(-1), b)]
        d["p"].append(torch.full((ad[-1],), LOG_STD, device="cuda"))
        d["g"] = [0.01 * _normal(g, t.numel()) for t in d["p"]]
        d["m"] = [0.002 * _normal(g, t.numel()) for t in d["p"]]
        d["v"] = [1e-6 * (0.5 + torch.rand(t.numel(), generator=g, device="cuda")) for t in d["p"]]
    elif kind == "norm":
        dim = case["dim"]
        d["x"] = _normal(g, case["rows"], dim) * (0.5 + torch.rand(dim, generator=g, device="cuda")) + 0.5 + \
            0.1 * _normal(g, dim)
    else:  # grads, update
        n = case["rows"] if kind == "grads" else case["envs"] * case["steps"]
        d["obs"] = _obs(g, n, ad[0])
        d["cobs"] = d["obs"] if ad[0] == cd[0] else _obs(g, n, cd[0])
        d.update(_rollout(g, d["actor"], d["critic"], d["obs"], d["cobs"], ad[-1]))
    return d


def _config(case):
    common = dict(clip=CLIP, entropy_coef=ENTROPY, value_coef=VALUE_COEF, max_grad_norm=1.0)
    if case["kind"] == "grads":
        return PpoConfig(epochs=1, minibatches=1, **common)
    # A fixed learning rate and no early stop: every pass does the same work.
    common.update(epochs=case["epochs"], minibatches=case["minibatches"], adaptive_lr=False)
    return PpoConfig.gpu_trainer(early_stop=False, **common) if case["trainer"] else PpoConfig(shuffle=True, **common)


def _handle(d, rows):
    ac = GpuActorCritic(_ctx(), d["ad"], d["cd"], rows)
    ac.set_params(_packed(d["actor"]), _packed(d["critic"]), np.full(d["ad"][-1], LOG_STD, np.float32), 3e-4)
    return ac


def prepare(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    s = {"case": case, "kind": kind}
    if kind == "act":
        n, A = case["envs"], d["ad"][-1]
        ac = _handle(d, min(n, 24576))
        for key, norm in (("obs", ac.obs_norm), ("cobs", ac.critic_norm)):
            norm.buf.upload(d[key + "_state"].cpu().numpy())
        s.update(ac=ac, obs=Buf(d["obs"]), cobs=Buf(d["cobs"]), eps=Buf(d["eps"]), action=_new(n, A), logp=_new(n),
                 mean=_new(n, A), value=_new(n))
    elif kind == "returns":
        T, N = case["steps"], case["envs"]
        s["ac"] = _handle(d, max(1, T * N // 4))
        s["obs"], s["ld"] = _rows(d["obs"], case["pad"])
        s["boot"], _ = _rows(d["boot"], case["pad"])
        s.update(rewards=Buf(d["rewards"]), dones=Buf(d["dones"]), values=_new(T, N), last=_new(N), adv=_new(T, N),
                 ret=_new(T, N))
    elif kind == "layers":
        i, m, o, n = case["in"], case["mid"], case["out"], case["rows"]
        s.update({k: Buf(d[k]) for k in ("x", "w1", "b1", "w2", "b2", "g2")})
        s.update(y=_new(m, n), z=_new(o, n))
        if case["train"]:
            s.update(g1=_new(m, n), gx=_new(i, n), dw1=_new(m, i), db1=_new(m), dw2=_new(o, m), db2=_new(o))
    elif kind == "loss":
        n, A = case["rows"], case["actions"]
        f = (lambda x: Buf(x.t().contiguous())) if case["feature_major"] else Buf
        s.update({k: f(d[k]) for k in ("mean", "action", "mean_old")})
        s.update({k: Buf(d[k]) for k in ("log_std", "adv", "logp_old", "v", "value_old", "ret")})
        s.update(d_mean=_new(A, n) if case["feature_major"] else _new(n, A), d_log_std=_new(A), stats=_new(2), d_v=_new(n),
                 v_stat=_new(1))
    elif kind == "adam":
        for k in ("p", "g", "m", "v"):
            s[k] = [Buf(t.clone()) for t in d[k]]
        s["tensors"] = [(s["p"][j], s["g"][j], s["m"][j], s["v"][j], t.numel()) for j, t in enumerate(d["p"])]
        s.update(scale=_new(1), norm=_new(1))
    elif kind == "norm":
        dim = case["dim"]
        s["x"], s["ld"] = _rows(d["x"], case["pad"])
        s.update(live=GpuNormalizer(_ctx(), dim), pending=GpuPendingNorm(_ctx(), dim), out=_new(case["rows"], dim))
        # The states live in torch memory, so that the outputs are tensors.
        for k in ("live", "pending"):
            s[k].buf = Buf(torch.from_numpy(s[k].buf.numpy()).cuda())
    else:
        n = d["obs"].shape[0]
        s.update(ac=_handle(d, n if kind == "grads" else max(1, n // case["minibatches"])),
                 batch=Batch(d, case["feature_major"]), cfg=_config(case))
    return s


def run(s):
    c, kind, case = _ctx(), s["kind"], s["case"]
    if kind == "act":
        ac = s["ac"]
        ac.act(s["obs"], case["envs"], s["eps"], s["action"], s["logp"], mean=s["mean"], value=s["value"],
               critic_obs=s["cobs"], obs_norm=ac.obs_norm, critic_norm=ac.critic_norm)
        return [s[k].tensor for k in ("action", "logp", "mean", "value")]
    if kind == "returns":
        T, N = case["steps"], case["envs"]
        s["ac"].values(s["obs"], T * N, s["values"], ld=s["ld"])
        s["ac"].values(s["boot"], N, s["last"], ld=s["ld"])
        ops.gae(c, s["rewards"], s["values"], s["dones"], s["last"], T, N, s["adv"], s["ret"], GAMMA, LAM)
        ops.adv_normalize(c, s["adv"], T * N)
        return [s[k].tensor for k in ("values", "last", "adv", "ret")]
    if kind == "layers":
        i, m, o, n = case["in"], case["mid"], case["out"], case["rows"]
        ops.gemm_bias_act(c, s["y"], s["w1"], s["x"], m, n, i, s["b1"], 1, True)
        ops.gemm_bias_act(c, s["z"], s["w2"], s["y"], o, n, m, s["b2"], 1, False)
        if not case["train"]:
            return [s["y"].tensor, s["z"].tensor]
        ops.gemm(c, s["dw2"], s["g2"], False, s["y"], True, o, m, n)
        ops.row_sum(c, s["db2"], s["g2"], o, n)
        ops.gemm(c, s["g1"], s["w2"], True, s["g2"], False, m, n, o)
        ops.elu_backward(c, s["g1"], s["y"], m, n)
        ops.gemm(c, s["dw1"], s["g1"], False, s["x"], True, m, i, n)
        ops.row_sum(c, s["db1"], s["g1"], m, n)
        ops.gemm(c, s["gx"], s["w1"], True, s["g1"], False, i, n, m)
        return [s[k].tensor for k in ("y", "z", "dw2", "db2", "g1", "dw1", "db1", "gx")]
    if kind == "loss":
        n, A = case["rows"], case["actions"]
        ops.ppo_actor_grad(c, s["mean"], s["action"], s["log_std"], s["adv"], s["logp_old"], s["mean_old"], n, A, CLIP,
                           ENTROPY, 1.0 / n, s["d_mean"], s["d_log_std"], s["stats"], feature_major=case["feature_major"])
        ops.ppo_value_grad(c, s["v"], s["value_old"], s["ret"], n, CLIP, VALUE_COEF, 1.0 / n, s["d_v"], s["v_stat"])
        return [s[k].tensor for k in ("d_mean", "d_log_std", "stats", "d_v", "v_stat")]
    if kind == "adam":
        ops.adam_multi_clip(c, s["tensors"], 1e-3, 1.0 - BETA1 ** 11, 1.0 - BETA2 ** 11, case["max_norm"], s["scale"],
                            s["norm"])
        return [[b.tensor for b in s[k]] for k in ("p", "m", "v")] + [s["scale"].tensor, s["norm"].tensor]
    if kind == "norm":
        s["pending"].push(s["x"], case["rows"], s["ld"])
        s["live"].commit(s["pending"])
        s["live"].normalize(s["x"], case["rows"], s["out"], ld_x=s["ld"])
        return [s["live"].buf.tensor, s["out"].tensor]
    if kind == "grads":
        ga, gc, gl, st = s["ac"].minibatch_grads(s["batch"], s["cfg"], 0, case["rows"])
        return [ga, gc, gl, st["surrogate"], st["value_loss"], st["kl"]]
    st = s["ac"].update(s["batch"], s["cfg"])
    a, cr, ls, lr = s["ac"].get_params()
    return [a, cr, ls, lr, st.value_loss, st.entropy]


# -------------------------------------------------------------------- work

def _macs(text):
    d = _dims(text)
    return sum(d[i] * d[i + 1] for i in range(len(d) - 1))


def _params(text):
    d = _dims(text)
    return sum(d[i] * d[i + 1] + d[i + 1] for i in range(len(d) - 1))


def work(case):
    kind = case["kind"]
    if kind in ("act", "returns", "grads", "update", "adam"):
        a, c = case["actor"], case["critic"]
        od, cd, A = _dims(a)[0], _dims(c)[0], _dims(a)[-1]
        macs, par = _macs(a) + _macs(c), _params(a) + _params(c)
        # Forward and weight gradient of every layer, data gradient of all but the first.
        step = 2 * (3 * macs - _dims(a)[0] * _dims(a)[1] - _dims(c)[0] * _dims(c)[1])
        row = od + (0 if od == cd else cd) + 2 * A + 4
    if kind == "act":
        n = case["envs"]
        return {"bytes": 4.0 * (n * (od + cd + 3 * A + 2) + par), "flops": 2.0 * n * macs}
    if kind == "returns":
        n = case["envs"] * case["steps"]
        return {"bytes": 4.0 * ((n + case["envs"]) * (cd + 1) + 3 * n + _params(c)) + n,
                "flops": 2.0 * (n + case["envs"]) * _macs(c)}
    if kind == "layers":
        i, m, o, n = case["in"], case["mid"], case["out"], case["rows"]
        if case["train"]:
            return {"bytes": 4.0 * (n * (2 * i + 2 * m + 2 * o) + 2 * (i * m + m * o + m + o)),
                    "flops": 6.0 * n * (i * m + m * o)}
        return {"bytes": 4.0 * (n * (i + m + o) + i * m + m * o + m + o), "flops": 2.0 * n * (i * m + m * o)}
    if kind == "loss":
        n, A = case["rows"], case["actions"]
        return {"bytes": 4.0 * (n * (4 * A + 6) + 2 * A), "flops": 30.0 * n * A}
    if kind == "adam":
        return {"bytes": 28.0 * (par + A), "flops": 16.0 * (par + A)}
    if kind == "norm":
        n = case["rows"] * case["dim"]
        return {"bytes": 8.0 * n, "flops": 8.0 * n}
    if kind == "grads":
        return {"bytes": 4.0 * (case["rows"] * row + 2 * par), "flops": float(step * case["rows"])}
    mb = case["envs"] * case["steps"] // case["minibatches"]
    n = case["epochs"] * mb * case["minibatches"]
    # The rows of every minibatch and the parameters with their moments at every step.
    return {"bytes": 4.0 * (n * row + 6 * par * case["epochs"] * case["minibatches"]), "flops": float(step * n)}


def tolerance(case):
    kind = case["kind"]
    if kind == "update":
        # Tens of Adam steps: a component whose gradient is near zero moves by
        # the learning rate in a direction that the last bit decides, and the
        # clipped objective amplifies it.
        return {"rel": 2e-2, "max": 0.15}
    if kind == "grads":
        # The probability ratio is the exponential of a difference of sums of
        # tens, so fp32 leaves 1e-5 of the gradients open.
        return {"rel": 5e-5, "max": 2e-3}
    return {"rel": 1e-5, "max": 1e-4}


# -------------------------------------------------------- float64 results

def _loss_grads(d, mean, v, n):
    """dL/dmean, dL/dlog_std, dL/dv and the three statistics, float64."""
    x = {k: d[k].double() for k in ("action", "mean_old", "logp_old", "value_old", "adv", "ret", "log_std")}
    ls, a = x["log_std"], x["adv"]
    diff = x["action"] - mean
    ratio = torch.exp(_logp(x["action"], mean, ls) - x["logp_old"])
    surr = torch.minimum(ratio * a, torch.clamp(ratio, 1 - CLIP, 1 + CLIP) * a)
    clipped = ((a >= 0) & (ratio > 1 + CLIP)) | ((a < 0) & (ratio < 1 - CLIP))
    coef = torch.where(clipped, torch.zeros_like(a), a * ratio)[:, None]
    inv_var = torch.exp(-2 * ls)
    d_mean = -coef * diff * inv_var / n
    d_ls = (-coef * (diff * diff * inv_var - 1) / n).sum(0) - ENTROPY
    kl = (0.5 * ((mean - x["mean_old"]) * torch.exp(-ls)) ** 2).sum() / n
    vc = x["value_old"] + torch.clamp(v - x["value_old"], -CLIP, CLIP)
    lu, lc = (v - x["ret"]) ** 2, (vc - x["ret"]) ** 2
    d_v = VALUE_COEF * 2 * torch.where(lc > lu, vc - x["ret"], v - x["ret"]) / n
    return d_mean, d_ls, d_v, surr.sum() / n, torch.maximum(lc, lu).sum() / n, kl


def _backward(net, acts, g):
    """Packed gradients of a network for dL/dout = g."""
    out = []
    for i in range(len(net) - 1, -1, -1):
        out = [(g.t() @ acts[i]).reshape(-1), g.sum(0)] + out
        if i:
            y = acts[i]
            g = (g @ net[i][0]) * torch.where(y > 0, torch.ones_like(y), y + 1)
    return torch.cat(out)


def exact(case, seed):
    kind = case["kind"]
    if kind == "update":
        return None  # tens of dependent steps: fp32 results scatter around any other precision's
    d = _inputs(case, seed)
    if kind == "act":
        outs = []
        for key, net in (("obs", d["actor"]), ("cobs", d["critic"])):
            st = d[key + "_state"].double()
            dim = d[key].shape[1]
            sd = torch.sqrt(torch.clamp(st[dim:2 * dim] / st[-1], min=1e-8))
            outs.append(_forward(_double(net), torch.clamp((d[key].double() - st[:dim]) / sd, -5, 5))[-1])
        ls = torch.full((d["ad"][-1],), LOG_STD, device="cuda", dtype=torch.float64)
        action = outs[0] + torch.exp(ls) * d["eps"].double()
        return [action, _logp(action, outs[0], ls), outs[0], outs[1][:, 0]]
    if kind == "returns":
        T, N = case["steps"], case["envs"]
        net = _double(d["critic"])
        v = torch.cat([_forward(net, x.double())[-1] for x in d["obs"].split(32768)])[:, 0].reshape(T, N)
        last = _forward(net, d["boot"].double())[-1][:, 0]
        adv, acc, nxt = torch.empty_like(v), torch.zeros_like(last), last
        for t in range(T - 1, -1, -1):
            live = 1.0 - d["dones"][t].double()
            acc = d["rewards"][t].double() + GAMMA * nxt * live - v[t] + GAMMA * LAM * live * acc
            adv[t], nxt = acc, v[t]
        norm = (adv - adv.mean()) / torch.clamp(adv.std(unbiased=False), min=1e-6)
        return [v, last, norm, adv + v]
    if kind == "layers":
        x, w1, b1, w2, b2, g2 = (d[k].double() for k in ("x", "w1", "b1", "w2", "b2", "g2"))
        z1 = w1 @ x + b1[:, None]
        y = torch.where(z1 > 0, z1, torch.expm1(torch.clamp(z1, max=0.0)))
        z = w2 @ y + b2[:, None]
        if not case["train"]:
            return [y, z]
        g1 = (w2.t() @ g2) * torch.where(y > 0, torch.ones_like(y), y + 1)
        return [y, z, g2 @ y.t(), g2.sum(1), g1, g1 @ x.t(), g1.sum(1), w1.t() @ g1]
    if kind == "loss":
        dm, dl, dv, surr, vl, kl = _loss_grads(d, d["mean"].double(), d["v"].double(), case["rows"])
        return [dm.t().contiguous() if case["feature_major"] else dm, dl, torch.stack([surr, kl]), dv, vl.reshape(1)]
    if kind == "adam":
        norm = math.sqrt(sum(float((t.double() ** 2).sum()) for t in d["g"]))
        scale = case["max_norm"] / norm if norm > case["max_norm"] else 1.0
        # The library takes its scalars as fp32.
        f = lambda x: float(np.float32(x))  # noqa: E731
        b1, b2, lr, eps, bc1, bc2 = f(BETA1), f(BETA2), f(1e-3), f(EPS), f(1 - BETA1 ** 11), f(1 - BETA2 ** 11)
        P, M, V = [], [], []
        for p, gr, m, v in zip(d["p"], d["g"], d["m"], d["v"]):
            gr = gr.double() * scale
            M.append(b1 * m.double() + (1 - b1) * gr)
            V.append(b2 * v.double() + (1 - b2) * gr * gr)
            P.append(p.double() - lr * (M[-1] / bc1) / (torch.sqrt(V[-1] / bc2) + eps))
        one = lambda x: torch.tensor([x], dtype=torch.float64)  # noqa: E731
        return [P, M, V, one(scale), one(norm)]
    if kind == "norm":
        x = d["x"].double()
        n, dim = x.shape
        mean, m2 = x.mean(0), ((x - x.mean(0)) ** 2).sum(0)
        # A new normaliser holds one observation's worth of prior: mean 0, m2 1, count 1.
        tot = n + 1.0
        m2 = 1.0 + m2 + mean * mean * n / tot
        mean = mean * n / tot
        out = torch.clamp((x - mean) / torch.sqrt(torch.clamp(m2 / tot, min=1e-8)), -5, 5)
        return [torch.cat([mean, m2, torch.tensor([tot], device="cuda", dtype=torch.float64)]), out]
    # grads
    n = case["rows"]
    nets = (_double(d["actor"]), _double(d["critic"]))
    acts = (_forward(nets[0], d["obs"].double()), _forward(nets[1], d["cobs"].double()))
    dm, dl, dv, surr, vl, kl = _loss_grads(d, acts[0][-1], acts[1][-1][:, 0], n)
    return [_backward(nets[0], acts[0], dm), _backward(nets[1], acts[1], dv[:, None]), dl, float(surr), float(vl),
            float(kl)]
