"""The calls a user of ppo_amd makes, as measurable cases.

Every case is one pass through a public entry point of the package: the
advantages of a rollout (gae_normalize, gae), the PPO losses of a minibatch
with their backward (ppo_loss_discrete, ppo_loss_gaussian), action selection
for a vector of environments (mlp_act_categorical), the gradients of one
minibatch through the actor and critic MLPs (ppo_mlp_cat_grads), and a whole
update of a rollout (VecPPO.update).  listed() holds the sizes of the
package's own benchmark together with small, odd and large ones; draw() gives
more of the same ranges; exact() restates each path in 64-bit torch or numpy.
"""

import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "zero-to-hero_amd"))
import ppo_amd  # noqa: E402

GAMMA, LAM, EPS = 0.99, 0.95, 1e-8
CLIP, VF_CLIP, VALUE_COEF, ENTROPY_COEF = 0.2, 0.2, 0.5, 0.01


def listed():
    return [
        # one CartPole iteration's rollout, the reference's environment with 8
        # copies: the smallest call, launches and latency
        dict(name="gae_128x8", path="gae", T=128, N=8, norm=True, bootstrap=True),
        # a classic-control rollout of the update-loop benchmark
        dict(name="gae_2048x64", path="gae", T=2048, N=64, norm=True, bootstrap=True),
        # the headline benchmark's rollout: 4096 environments on one GPU
        dict(name="gae_2048x4096", path="gae", T=2048, N=4096, norm=True, bootstrap=True),
        # a long horizon of few environments, advantages not normalised
        dict(name="gae_1048576x16", path="gae", T=1048576, N=16, norm=False, bootstrap=False),
        # an environment count that no vector width divides
        dict(name="gae_1000x1023", path="gae", T=1000, N=1023, norm=True, bootstrap=True),
        # the headline benchmark's loss: all samples of that rollout, the 18
        # actions of the full Atari set, forward and backward
        dict(name="cat_8388608x18", path="cat", B=8388608, A=18, vclip=True, int64=False),
        # a 4-action policy (LunarLander-sized) over an odd number of samples,
        # int64 actions as torch's sampling gives them
        dict(name="cat_100003x4", path="cat", B=100003, A=4, vclip=False, int64=True),
        # a large discrete action set (tokens, board moves)
        dict(name="cat_262144x64", path="cat", B=262144, A=64, vclip=True, int64=False),
        # continuous control: the Gaussian loss of the benchmark, 6 dimensions
        dict(name="gauss_2097152x6", path="gauss", B=2097152, D=6, vclip=False),
        # one action-selection step for 4096 environments
        dict(name="act_4096", path="act", N=4096, D=8, H=64, A=4, act="tanh"),
        # one large minibatch through the reference's 128-wide ReLU networks
        dict(name="mlp_32768", path="mlp", B=32768, D=8, H=128, A=4, act="relu", vclip=False),
        # a whole update of the CartPole configuration: 4 epochs of 4
        # minibatches of 256, 4-64-64 tanh networks, replayed from graphs
        dict(name="update_128x8", path="update", T=128, N=8, mb=256, D=4, H=64, A=2,
             act="tanh"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["gae", "gae", "cat", "cat", "gauss", "act", "mlp", "update"])
    flag = lambda: rng.random() < 0.5  # noqa: E731
    if path == "gae":
        N = _log_int(rng, 1, 4096)
        T = _log_int(rng, 16, min(1048576, (1 << 24) // N))
        if flag():  # environment counts are often multiples of 8
            N = max(8, N // 8 * 8)
        return dict(path=path, T=T, N=N, norm=flag(), bootstrap=flag())
    if path == "cat":
        A = _log_int(rng, 2, 128)
        return dict(path=path, B=_log_int(rng, 64, (1 << 25) // A), A=A, vclip=flag(),
                    int64=flag())
    if path == "gauss":
        D = _log_int(rng, 1, 24)
        return dict(path=path, B=_log_int(rng, 64, (1 << 24) // D), D=D, vclip=flag())
    net = dict(H=rng.choice([16, 32, 64, 128]), act=rng.choice(["tanh", "relu"]),
               D=_log_int(rng, 2, 64), A=_log_int(rng, 2, 18))
    if path == "act":
        return dict(path=path, N=_log_int(rng, 1, 16384), **net)
    if path == "mlp":
        return dict(path=path, B=_log_int(rng, 64, 32768), vclip=flag(), **net)
    N, mb = rng.randint(1, 32), rng.choice([64, 128, 256, 512])
    return dict(path=path, T=max(16, min(_log_int(rng, 2 * mb, 8 * mb), 4096) // N), N=N, mb=mb,
                **net)


# --- inputs, from the seed alone ------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * seed + 17)
    return g


def _rn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _ru(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda")


def _rollout_inputs(case, seed):
    """Rewards and values of order 1, an episode end about every 100 steps."""
    g, T, N = _gen(seed), case["T"], case["N"]
    r, v = _rn(g, T, N), _rn(g, T, N)
    d = (_ru(g, T, N) < 0.01).to(torch.uint8)
    return r, v, d, _rn(g, N) if case["bootstrap"] else None


def _row_inputs(g, lp, v, vclip):
    """The per-sample inputs beside a policy's log-probs lp and values v: old
    log-probs of a policy some updates ago, normalised advantages, returns and
    old values.  The loss's gradient jumps at the clip bounds; samples closer to
    one than fp32 arithmetic resolves are moved off it, so that every correct
    implementation puts them on the same side."""
    B = lp.numel()
    adv = _rn(g, B)
    # new minus old log-prob: ratios around 1, larger where the advantage is
    shift = -0.02 + 0.05 * adv + 0.13 * _rn(g, B)
    ratio = shift.exp()
    near = ((ratio - (1 + CLIP)).abs() < 2e-4) | ((ratio - (1 - CLIP)).abs() < 2e-4)
    old_lp = lp - torch.where(near, shift + 1e-3, shift)
    old_v = v - 0.15 * _rn(g, B)
    off = ((v - old_v).abs() - VF_CLIP).abs() < 1e-3
    old_v = torch.where(off, old_v - 5e-3, old_v)
    ret = v + 0.5 * _rn(g, B)
    if vclip:
        vc = old_v + (v - old_v).clamp(-VF_CLIP, VF_CLIP)
        out = (v - old_v).abs() > VF_CLIP
        tie = ((v - vc) * (v + vc - 2 * ret)).abs() < 1e-5 * (1 + (v - ret) ** 2)
        ret = torch.where(out & tie, ret + 0.1, ret)
    return old_lp.contiguous(), adv, ret.contiguous(), old_v.contiguous()


def _cat_inputs(case, seed):
    g, B, A = _gen(seed), case["B"], case["A"]
    logits, v = _rn(g, B, A), _rn(g, B)
    # actions drawn from the policy (Gumbel maximum), in slices to bound memory
    act = torch.empty(B, dtype=torch.int64, device="cuda")
    lp = torch.empty(B, device="cuda")
    for i in range(0, B, 1 << 20):
        z = logits[i:i + (1 << 20)]
        u = _ru(g, *z.shape).clamp_(1e-20, 1 - 1e-7)
        act[i:i + (1 << 20)] = (z - (-u.log()).log()).argmax(1)
        lp[i:i + (1 << 20)] = z.log_softmax(1).gather(1, act[i:i + (1 << 20), None]).squeeze(1)
    rows = _row_inputs(g, lp, v, case["vclip"])
    return logits, (act if case["int64"] else act.to(torch.int32)), v, rows


def _gauss_inputs(case, seed):
    g, B, D = _gen(seed), case["B"], case["D"]
    mu, v = _rn(g, B, D), _rn(g, B)
    log_std = -0.5 + 0.1 * _rn(g, D)
    act = mu + log_std.exp() * _rn(g, B, D)
    lp = (-(act.double() - mu.double()) ** 2 / (2 * (2 * log_std.double()).exp())
          - log_std.double() - 0.5 * math.log(2 * math.pi)).sum(1).float()
    return mu, log_std, act, v, _row_inputs(g, lp, v, case["vclip"])


def _weights(g, D, H, O):
    """nn.Linear's initial distribution for a D-H-H-O network, from g."""
    sizes, got = [(D, H), (H, H), (H, O)], []
    for i, o in sizes:
        k = 1.0 / math.sqrt(i)
        got += [(2 * _ru(g, o, i) - 1) * k, (2 * _ru(g, o) - 1) * k]
    return got


def _net(case, weights, O):
    net = ppo_amd.MLP(case["D"], case["H"], O, activation=case["act"]).to("cuda")
    with torch.no_grad():
        for p, w in zip(net.parameters(), weights):
            p.copy_(w)
    return net


def _forward64(weights, x, act, hidden=False):
    f = torch.tanh if act == "tanh" else torch.relu
    w = [t.double() if t.dtype != torch.float64 else t for t in weights]
    a = F.linear(x.double(), w[0], w[1])
    b = F.linear(f(a), w[2], w[3])
    return (a, b) if hidden else F.linear(f(b), w[4], w[5])


def _policy_inputs(g, case, n):
    """Both networks' weights, n observations, and for each the action drawn from
    the policy, its log-prob and the critic's value.  Observations that put a ReLU
    closer to its kink than fp32 resolves are scaled a little, for the reason given
    in _row_inputs."""
    wa, wc = _weights(g, case["D"], case["H"], case["A"]), _weights(g, case["D"], case["H"], 1)
    obs = _rn(g, n, case["D"])
    for _ in range(3 if case["act"] == "relu" else 0):
        pre = torch.cat([t for w in (wa, wc) for t in _forward64(w, obs, "relu", True)], 1)
        obs = torch.where((pre.abs().amin(1) < 1e-6)[:, None], obs * 1.01, obs)
    z = _forward64(wa, obs, case["act"])
    u = _ru(g, *z.shape).double().clamp_(1e-20, 1 - 1e-7)
    act = (z - (-u.log()).log()).argmax(1)
    lp = z.log_softmax(1).gather(1, act[:, None]).squeeze(1).float()
    v = _forward64(wc, obs, case["act"]).squeeze(1).float()
    return wa, wc, obs, act.to(torch.int32), lp, v


def _act_inputs(case, seed):
    """Uniforms nearer to a boundary between two actions than fp32 resolves move to
    the middle of the likeliest action."""
    g, N = _gen(seed), case["N"]
    wa, wc, obs, _, _, _ = _policy_inputs(g, case, N)
    p = _forward64(wa, obs, case["act"]).softmax(1)
    cdf = p.cumsum(1)
    u = _ru(g, N)
    near = (cdf - u.double()[:, None]).abs().amin(1) < 1e-5
    best = p.argmax(1, keepdim=True)
    mid = (cdf - p / 2).gather(1, best).squeeze(1).float()
    return wa, wc, obs, torch.where(near, mid, u)


def _mlp_inputs(case, seed):
    """A rollout of B samples visited in a shuffled order."""
    g = _gen(seed)
    wa, wc, obs, act, lp, v = _policy_inputs(g, case, case["B"])
    rows = _row_inputs(g, lp, v, case["vclip"])
    return wa, wc, obs, act, rows, torch.randperm(case["B"], generator=g, device="cuda")


def _update_inputs(case, seed):
    """A rollout collected with the networks as they are: reward 1 a step, an
    episode end about every 50 steps."""
    g, n = _gen(seed), case["T"] * case["N"]
    wa, wc, obs, act, lp, v = _policy_inputs(g, case, n)
    d = (_ru(g, n) < 0.02).to(torch.uint8)
    return wa, wc, obs, act, lp, v, d, _rn(g, case["N"])


# --- what a program has in hand before the call ---------------------------------------

def prepare(case, seed):
    path = case["path"]
    s = {"case": case}
    if path == "gae":
        s["r"], s["v"], s["d"], s["lv"] = _rollout_inputs(case, seed)
    elif path == "cat":
        logits, s["act"], v, s["rows"] = _cat_inputs(case, seed)
        s["logits"], s["v"] = logits.requires_grad_(), v.requires_grad_()
    elif path == "gauss":
        mu, log_std, s["act"], v, s["rows"] = _gauss_inputs(case, seed)
        s["mu"], s["log_std"], s["v"] = (t.requires_grad_() for t in (mu, log_std, v))
    elif path == "act":
        wa, wc, s["obs"], s["u"] = _act_inputs(case, seed)
        s["policy"], s["value"] = _net(case, wa, case["A"]), _net(case, wc, 1)
    elif path == "mlp":
        wa, wc, s["obs"], s["act"], s["rows"], s["idx"] = _mlp_inputs(case, seed)
        s["policy"], s["value"] = _net(case, wa, case["A"]), _net(case, wc, 1)
    else:
        T, N = case["T"], case["N"]
        wa, wc, obs, act, lp, v, d, lv = _update_inputs(case, seed)
        s["policy"], s["value"] = _net(case, wa, case["A"]), _net(case, wc, 1)
        s["ppo"] = ppo_amd.VecPPO(s["policy"], s["value"], batch_size=case["mb"], graphs=True,
                                  generator=torch.Generator().manual_seed(seed))
        b = s["buffer"] = ppo_amd.RolloutBuffer(T, N, (case["D"],))
        for t in range(T):
            i = slice(t * N, (t + 1) * N)
            b.add(obs[i], act[i], torch.ones(N, device="cuda"), d[i], v[i], lp[i])
        b.finish(lv)
    return s


# The loss's reported scalars, without approx_kl: a mean of differences of nearly
# equal log-probs, whose leading digits cancel, so that its last ones are rounding
# that no two orders of summation share.
SCALARS = ("loss", "policy", "value", "entropy", "clipfrac")


def _scalars(stats, names=SCALARS):
    return {k: stats[k] for k in names}


def run(s):
    c = s["case"]
    path = c["path"]
    if path == "gae":
        if c["norm"]:
            return ppo_amd.gae_normalize(s["r"], s["v"], s["d"], s["lv"], GAMMA, LAM)
        return ppo_amd.gae(s["r"], s["v"], s["d"], s["lv"], GAMMA, LAM)
    if path == "cat":
        s["logits"].grad = s["v"].grad = None
        old_lp, adv, ret, old_v = s["rows"]
        loss, stats = ppo_amd.ppo_loss_discrete(
            s["logits"], s["act"], old_lp, adv, ret, s["v"], old_v if c["vclip"] else None,
            CLIP, VF_CLIP if c["vclip"] else None, VALUE_COEF, ENTROPY_COEF)
        loss.backward()
        return {"stats": _scalars(stats), "dlogits": s["logits"].grad, "dvalues": s["v"].grad}
    if path == "gauss":
        s["mu"].grad = s["log_std"].grad = s["v"].grad = None
        old_lp, adv, ret, old_v = s["rows"]
        loss, stats = ppo_amd.ppo_loss_gaussian(
            s["mu"], s["log_std"], s["act"], old_lp, adv, ret, s["v"],
            old_v if c["vclip"] else None, CLIP, VF_CLIP if c["vclip"] else None, VALUE_COEF,
            ENTROPY_COEF)
        loss.backward()
        return {"stats": _scalars(stats), "dmu": s["mu"].grad, "dlog_std": s["log_std"].grad,
                "dvalues": s["v"].grad}
    if path == "act":
        return ppo_amd.mlp_act_categorical(s["policy"], s["value"], s["obs"], uniforms=s["u"])
    if path == "mlp":
        old_lp, adv, ret, old_v = s["rows"]
        stats = ppo_amd.ppo_mlp_cat_grads(
            s["policy"], s["value"], s["obs"], s["act"], old_lp, adv, ret,
            old_v if c["vclip"] else None, s["idx"], CLIP, VF_CLIP if c["vclip"] else None,
            VALUE_COEF, ENTROPY_COEF)
        return {"stats": _scalars(stats), "policy": [p.grad for p in s["policy"].parameters()],
                "value": [p.grad for p in s["value"].parameters()]}
    stats = s["ppo"].update(s["buffer"])
    # (the last minibatch's policy loss is a mean near zero: not compared)
    return {"stats": _scalars(stats, ("loss", "value", "entropy")),
            "policy": [p.detach() for p in s["policy"].parameters()],
            "value": [p.detach() for p in s["value"].parameters()]}


# --- what a pass cannot do without ----------------------------------------------------

def _params(c):
    D, H, A = c["D"], c["H"], c["A"]
    return 2 * (D * H + H + H * H + H) + (A + 1) * (H + 1)


def work(case):
    c, path = case, case["path"]
    if path == "gae":  # rewards, values, dones in; advantages, returns (and normalised) out
        return {"bytes": c["T"] * c["N"] * (9 + (12 if c["norm"] else 8)),
                "flops": 10 * c["T"] * c["N"]}
    if path == "cat":  # logits, action, 4-5 row arrays in; both gradients out
        row = 8 * c["A"] + (8 if c["int64"] else 4) + (20 if c["vclip"] else 16) + 4
        return {"bytes": c["B"] * row, "flops": 12 * c["B"] * c["A"]}
    if path == "gauss":
        return {"bytes": c["B"] * (12 * c["D"] + (20 if c["vclip"] else 16) + 4),
                "flops": 12 * c["B"] * c["D"]}
    if path == "act":
        return {"bytes": c["N"] * (4 * c["D"] + 16) + 4 * _params(c),
                "flops": 2 * c["N"] * _params(c)}
    if path == "mlp":  # observations, index, 5-6 row arrays, weights in; gradients out
        return {"bytes": c["B"] * (4 * c["D"] + 8 + (20 if c["vclip"] else 16)) + 8 * _params(c),
                "flops": 6 * c["B"] * _params(c)}
    n = c["T"] * c["N"]
    steps = 4 * math.ceil(n / c["mb"])
    return {"bytes": n * 21 + 4 * n * (4 * c["D"] + 24) + steps * 24 * _params(c),
            "flops": 4 * n * 6 * _params(c)}


def tolerance(case):
    """About four times what the paths were seen to be off exact() by: fp32 rounding
    of each element (rollouts: 6e-8; softmax rows 2e-7; Gaussian rows, whose
    log-probs sum up to 24 squares, 8e-7), of sums over a minibatch (MLP gradients:
    2e-7), and over a whole update 1e-7 with smooth activations, more where a ReLU's
    kink falls between two roundings in a later step."""
    path = case["path"]
    if path == "gae":
        return {"rel": 3e-7}
    if path == "cat":
        return {"rel": 2e-6, "max": 1e-4}
    if path == "gauss":
        return {"rel": 5e-6, "max": 1e-4}
    if path == "act":
        return {"rel": 2e-6, "max": 1e-4, "differ": 1e-3}
    if path == "mlp":
        return {"rel": 2e-6, "max": 1e-4}
    return {"rel": 3e-5, "max": 1e-2}


# --- the same in 64 bits --------------------------------------------------------------

def _gae64(r, v, d, lv):
    T, N = r.shape
    dev = r.device
    if T > 4096:  # many short rows: numpy's loop on the host
        r, v, nd = (t.cpu().numpy().astype(np.float64) for t in (r, v, 1 - d.double()))
        nxt = np.zeros(N) if lv is None else lv.cpu().numpy().astype(np.float64)
        adv, x = np.empty((T, N)), np.zeros(N)
        for t in range(T - 1, -1, -1):
            x = r[t] + GAMMA * nxt * nd[t] - v[t] + GAMMA * LAM * nd[t] * x
            adv[t], nxt = x, v[t]
        return torch.from_numpy(adv).to(dev)
    r, v, nd = r.double(), v.double(), 1 - d.double()
    nxt = torch.zeros(N, dtype=torch.float64, device=dev) if lv is None else lv.double()
    delta = r + GAMMA * torch.cat([v[1:], nxt[None]]) * nd - v
    adv, x = torch.empty_like(delta), torch.zeros_like(nxt)
    for t in range(T - 1, -1, -1):
        x = delta[t] + GAMMA * LAM * nd[t] * x
        adv[t] = x
    return adv


def _normalize64(adv):
    return (adv - adv.mean()) / (adv.std() + EPS) if adv.numel() > 1 else adv


def _loss64(lp, entropy, rows, v, vclip, vf_clip=VF_CLIP):
    old_lp, adv, ret, old_v = (None if t is None else t.double() for t in rows)
    ratio = (lp - old_lp).exp()
    policy = -torch.minimum(ratio * adv, ratio.clamp(1 - CLIP, 1 + CLIP) * adv).mean()
    sq = (v - ret) ** 2
    if vclip:
        sq = torch.maximum(sq, (old_v + (v - old_v).clamp(-vf_clip, vf_clip) - ret) ** 2)
    value, ent = sq.mean(), entropy.mean()
    loss = policy + VALUE_COEF * value - ENTROPY_COEF * ent
    stats = {"loss": loss, "policy": policy, "value": value, "entropy": ent,
             "clipfrac": ((ratio - 1).abs() > CLIP).double().mean()}
    return loss, {k: t.detach() for k, t in stats.items()}


def _cat_terms64(z, act):
    logp = z.log_softmax(1)
    return logp.gather(1, act.long()[:, None]).squeeze(1), -(logp.exp() * logp).sum(1)


def _cat64(z, act, rows, v, vclip):
    return _loss64(*_cat_terms64(z, act), rows, v, vclip)


def _leaves64(weights):
    return [w.double().requires_grad_() for w in weights]


def exact(case, seed):
    path = case["path"]
    if path == "gae":
        r, v, d, lv = _rollout_inputs(case, seed)
        adv = _gae64(r, v, d, lv)
        return (adv, adv + v.double()) + ((_normalize64(adv),) if case["norm"] else ())
    if path == "cat":
        logits, act, v, rows = _cat_inputs(case, seed)
        z, v = logits.double().requires_grad_(), v.double().requires_grad_()
        loss, stats = _cat64(z, act, rows, v, case["vclip"])
        loss.backward()
        return {"stats": stats, "dlogits": z.grad, "dvalues": v.grad}
    if path == "gauss":
        mu, log_std, act, v, rows = _gauss_inputs(case, seed)
        mu, log_std, v = (t.double().requires_grad_() for t in (mu, log_std, v))
        lp = (-(act.double() - mu) ** 2 / (2 * (2 * log_std).exp()) - log_std
              - 0.5 * math.log(2 * math.pi)).sum(1)
        entropy = (0.5 + 0.5 * math.log(2 * math.pi) + log_std).sum().expand(mu.shape[0])
        loss, stats = _loss64(lp, entropy, rows, v, case["vclip"])
        loss.backward()
        return {"stats": stats, "dmu": mu.grad, "dlog_std": log_std.grad, "dvalues": v.grad}
    if path == "act":
        wa, wc, obs, u = _act_inputs(case, seed)
        logp = _forward64(wa, obs, case["act"]).log_softmax(1)
        act = (logp.exp().cumsum(1) <= u.double()[:, None]).sum(1).clamp(max=case["A"] - 1)
        return (act, logp.gather(1, act[:, None]).squeeze(1),
                _forward64(wc, obs, case["act"]).squeeze(1))
    if path == "mlp":
        wa, wc, obs, act, rows, idx = _mlp_inputs(case, seed)
        wa, wc = _leaves64(wa), _leaves64(wc)
        loss, stats = _cat64(_forward64(wa, obs[idx], case["act"]), act[idx],
                             tuple(t[idx] for t in rows),
                             _forward64(wc, obs[idx], case["act"]).squeeze(1), case["vclip"])
        loss.backward()
        return {"stats": stats, "policy": [p.grad for p in wa], "value": [p.grad for p in wc]}
    # a whole update: 4 epochs of clipped Adam steps on shuffled minibatches
    T, N, n = case["T"], case["N"], case["T"] * case["N"]
    wa, wc, obs, act, lp, v, d, lv = _update_inputs(case, seed)
    adv = _gae64(torch.ones(T, N, device="cuda"), v.view(T, N), d.view(T, N), lv)
    rows = (lp, _normalize64(adv).reshape(n), (adv + v.view(T, N).double()).reshape(n), v)
    wa, wc = _leaves64(wa), _leaves64(wc)
    params = wa + wc
    adam = torch.optim.Adam(params, lr=3e-4)
    perm_gen = torch.Generator().manual_seed(seed)
    perms = [torch.randperm(n, generator=perm_gen).to("cuda") for _ in range(4)]
    for perm in perms:
        for i in range(0, n, case["mb"]):
            idx = perm[i:i + case["mb"]]
            loss, stats = _cat64(_forward64(wa, obs[idx], case["act"]), act[idx],
                                 tuple(t[idx] for t in rows),
                                 _forward64(wc, obs[idx], case["act"]).squeeze(1), False)
            adam.zero_grad()
            loss.backward()
            torch.nn.utils.clip_grad_norm_(params, 0.5)
            adam.step()
    return {"stats": _scalars(stats, ("loss", "value", "entropy")),
            "policy": [p.detach() for p in wa],
            "value": [p.detach() for p in wc]}
