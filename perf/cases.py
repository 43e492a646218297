"""What a rollout worker does with this package, as cases that can be timed: generation (prompt cache fill and decode
steps) and the scoring pass through `TmxRollout`, and the LoRA weight sync between rollouts.

Shapes are those of `ModelConfig` with the quantisation and adapters `bench.py` gives them.  The 8B-class and MoE models
keep their widths and run a part of their depth (all layers are alike), so that a pass stays short; fewer tokens are
generated than a whole rollout has for the same reason.

Weights are `QLoRAModel.random_init`'s, with two things changed that a trained policy has and noise has not.  The
matrices that write to the residual stream are scaled down, so that the token just read still shows in the last hidden
state, and the head knows one successor for every token (tied embeddings: the token itself).  Next-token distributions
are therefore peaked: greedy cases choose with a clear margin and report log-probs of a few nats, sampled cases have one
token that takes nearly all of the mass.  With plain noise the two best of 128k logits are often closer than one bf16
step, and a sequence that once chose the other one never comes back.
"""
import dataclasses
import math

import numpy as np
import torch

from tunix_amd.configs import CacheConfig, RolloutConfig
from tunix_amd.model import ModelConfig, QLoRAModel
from tunix_amd.rollout import TmxRollout

ATTN = ('q_proj', 'k_proj', 'v_proj', 'o_proj')
MLP = ('gate_proj', 'up_proj', 'down_proj')
STD = 0.02  # random_init's standard deviation

# name -> (ModelConfig factory, group, LoRA rank, adapters)
MODELS = {
    'toy': ('toy', 64, 8, ATTN + MLP),
    'llama-1b': ('llama3p2_1b', 64, 16, ATTN + MLP),
    'llama-8b': ('llama3p1_8b', 64, 16, ATTN + MLP),
    'qwen-8b': ('qwen3_8b', 128, 32, ATTN + MLP),
    'qwen-30b-a3b': ('qwen3_30b_a3b', 64, 8, ATTN),
}


def _generate(name, model, layers, prompts, samples, shortest, longest, new, mode):
  return {'name': name, 'do': 'generate', 'model': model, 'layers': layers, 'prompts': prompts, 'samples': samples,
          'shortest': shortest, 'longest': longest, 'new': new, 'mode': mode}


def _score(name, model, layers, sequences, prompt, completion):
  return {'name': name, 'do': 'score', 'model': model, 'layers': layers, 'sequences': sequences, 'prompt': prompt,
          'completion': completion}


def _sync(name, model, layers, rank):
  return {'name': name, 'do': 'sync', 'model': model, 'layers': layers, 'rank': rank}


def listed():
  return [
      # the smallest model there is: unit tests, examples and dry runs of a training script; nothing but latency
      _generate('toy_greedy', 'toy', 2, 4, 1, 32, 32, 32, 'greedy'),
      # one sequence at a time: interactive use, the latency regime
      _generate('1b_single', 'llama-1b', 16, 1, 1, 256, 256, 64, 'sample'),
      # a small evaluation batch: prompts as long as they happen to be, greedy
      _generate('1b_eval_ragged', 'llama-1b', 16, 3, 1, 61, 250, 48, 'greedy'),
      # the GRPO rollout, the workload the package is benchmarked on: 8 samples of each of 8 prompts
      _generate('8b_grpo', 'llama-8b', 8, 8, 8, 256, 256, 64, 'sample'),
      # evaluation of the 8B model: a batch that is no power of two, ragged prompts, greedy
      _generate('8b_eval_ragged', 'llama-8b', 8, 23, 1, 17, 301, 32, 'greedy'),
      # more sequences than one decode block holds: a large GRPO batch
      _generate('8b_grpo_256', 'llama-8b', 8, 32, 8, 128, 128, 24, 'sample'),
      # long prompts, short answers (a judge or a classifier): all prompt
      _generate('8b_long_prompt', 'llama-8b', 8, 3, 1, 1021, 2040, 8, 'greedy'),
      # large batch of distinct prompts with nucleus sampling
      _generate('qwen_nucleus_128', 'qwen-8b', 6, 128, 1, 512, 512, 32, 'nucleus'),
      # routed experts, where a decode step reads nearly all of them
      _generate('moe_rollout_32', 'qwen-30b-a3b', 8, 32, 1, 256, 256, 48, 'sample'),
      # log-probs of the finished rollouts under the policy or the reference policy
      _score('8b_score', 'llama-8b', 8, 16, 256, 512),
      # the same for a handful of short sequences
      _score('1b_score_small', 'llama-1b', 16, 5, 37, 90),
      # the trainer's new adapters after every optimizer step
      _sync('8b_lora_sync', 'llama-8b', 8, 16),
  ]


def _log_int(rng, low, high):
  return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
  kind = rng.choice(['toy', '1b', '1b', '8b', '8b', 'grpo', 'grpo', 'long', 'qwen', 'moe', 'moe', 'score', 'score',
                     'score_small', 'sync'])
  mode = rng.choice(['greedy', 'sample'])
  if kind == 'toy':
    p = _log_int(rng, 5, 48)
    case = _generate('', 'toy', 2, rng.randint(1, 8), 1, max(1, p // rng.randint(1, 3)), p, _log_int(rng, 8, 48), mode)
  elif kind == '1b':
    p = _log_int(rng, 16, 512)
    case = _generate('', 'llama-1b', 16, rng.randint(1, 4), 1, max(4, p // rng.randint(1, 4)), p, _log_int(rng, 16, 64),
                     mode)
  elif kind == '8b':
    p = _log_int(rng, 24, 320)
    case = _generate('', 'llama-8b', 8, _log_int(rng, 5, 64), 1, max(4, p // rng.randint(1, 8)), p,
                     _log_int(rng, 8, 48), mode)
  elif kind == 'grpo':
    p = _log_int(rng, 48, 320)
    case = _generate('', 'llama-8b', 8, _log_int(rng, 2, 32), rng.randint(2, 8), p, p, _log_int(rng, 8, 48), 'sample')
  elif kind == 'long':
    p = _log_int(rng, 500, 2040)
    case = _generate('', 'llama-8b', 8, rng.randint(1, 3), 1, p // rng.randint(1, 2), p, rng.randint(2, 8), 'greedy')
  elif kind == 'qwen':
    p = _log_int(rng, 64, 500)
    case = _generate('', 'qwen-8b', 6, rng.randint(65, 128), 1, p // rng.randint(1, 3), p, _log_int(rng, 8, 32),
                     'nucleus')
  elif kind == 'moe':
    p = _log_int(rng, 32, 256)
    case = _generate('', 'qwen-30b-a3b', 8, _log_int(rng, 4, 32), 1, p // rng.randint(1, 3), p, _log_int(rng, 8, 48),
                     'sample')
  elif kind == 'score':
    case = _score('', 'llama-8b', 8, rng.randint(2, 16), _log_int(rng, 48, 256), _log_int(rng, 64, 512))
  elif kind == 'score_small':
    case = _score('', 'llama-1b', 16, rng.randint(1, 8), _log_int(rng, 16, 64), _log_int(rng, 24, 128))
  else:
    case = _sync('', rng.choice(['llama-1b', 'llama-8b', 'qwen-8b']), rng.randint(2, 8), rng.choice([8, 16, 32]))
  del case['name']
  return case


def _config(case):
  return dataclasses.replace(getattr(ModelConfig, MODELS[case['model']][0])(), num_layers=case['layers'])


class _Ids:
  """Tokenizer of a program that works on token ids: pad 0, bos 1, and no text."""

  def encode(self, text):
    return [int(t) for t in text.split()]

  def decode(self, ids):
    return ''

  def pad_id(self):
    return 0

  def bos_id(self):
    return 1

  def eos_id(self):
    return 2


def _lengths(n, shortest, longest, rng):
  """n prompt lengths spread evenly over the range, in an order of the seed's; the longest is always there."""
  spread = np.linspace(longest, shortest, n).round().astype(int)
  return rng.permutation(spread)


def _model(case, seed, rank=None):
  c = _config(case)
  _, group, default_rank, targets = MODELS[case['model']]
  rank = rank or default_rank
  m = QLoRAModel.random_init(c, seed=seed % (1 << 31), group=group, lora_rank=rank, lora_alpha=2.0 * rank,
                             lora_targets=targets, std=STD)
  # What a layer adds to the residual stream, from random_init's own scale: gate and up have the standard deviation `s`.
  s = STD * math.sqrt(c.embed_dim)
  mlp = STD * math.sqrt(c.hidden_dim) * 0.6 * s * s / math.sqrt(c.num_experts_per_tok or 1)
  attn = STD * math.sqrt(c.num_heads * c.head_dim) * 0.5 * s
  noise = math.sqrt(c.num_layers * (mlp * mlp + attn * attn))
  # The share of the embedding in the last hidden state.  A known successor's logit is share * STD * D, against a spread
  # of STD * sqrt(D) of the others: about 10 where choices are greedy and scores are compared, far above them elsewhere.
  share = min(0.6, 10.0 / (STD * c.embed_dim)) if case.get('mode', 'greedy') == 'greedy' else 0.95
  scale = STD * math.sqrt(1 - share * share) / share / noise
  for layer in m.layers:
    for key in ('o', 'down'):
      layer[key].scales.mul_(scale)
      if layer[key].lora_b is not None:
        layer[key].lora_b.mul_(scale)
  if not c.weight_tying:
    g = torch.Generator(device=m.device).manual_seed(seed % (1 << 31) + 1)
    m.head.copy_(m.embed[torch.randperm(c.vocab_size, generator=g, device=m.device)])
  return m


def _rollout(model, cache_size):
  c = model.config
  return TmxRollout(model, _Ids(), CacheConfig(cache_size, c.num_layers, c.num_kv_heads, c.head_dim))


def _adapters(config, rank, seed):
  """New adapters in the trainer's precision, as the nested state a weight sync is handed."""
  c = config
  g = torch.Generator(device='cuda').manual_seed(seed % (1 << 31))
  new = lambda *shape: torch.randn(*shape, generator=g, device='cuda') * STD
  d, f, n, kh, h = c.embed_dim, c.hidden_dim, c.num_heads, c.num_kv_heads, c.head_dim
  ins = {'q_proj': (d,), 'k_proj': (d,), 'v_proj': (d,), 'o_proj': (n, h), 'gate_proj': (d,), 'up_proj': (d,),
         'down_proj': (f,)}
  outs = {'q_proj': (n, h), 'k_proj': (kh, h), 'v_proj': (kh, h), 'o_proj': (d,), 'gate_proj': (f,), 'up_proj': (f,),
          'down_proj': (d,)}

  def part(names, w):
    return {p: {w + '_lora_a': new(*ins[p], rank), w + '_lora_b': new(rank, *outs[p])} for p in names}

  return {'layers': {i: {'attn': part(ATTN, 'w'), 'mlp': part(MLP, 'kernel')} for i in range(c.num_layers)}}


def prepare(case, seed):
  c = _config(case)
  rng = np.random.default_rng(seed)
  if case['do'] == 'sync':
    rollout = _rollout(_model(case, seed, case['rank']), 256)
    return {'do': 'sync', 'rollout': rollout, 'adapters': _adapters(c, case['rank'], seed + 7)}
  if case['do'] == 'score':
    b, p, t = case['sequences'], case['prompt'], case['completion']
    # prompts padded on the left, completions on the right, as a learner's batch is
    prompt = rng.integers(3, c.vocab_size, (b, p)).astype(np.int32)
    completion = rng.integers(3, c.vocab_size, (b, t)).astype(np.int32)
    for i, (np_, nt) in enumerate(zip(_lengths(b, (p + 1) // 2, p, rng), _lengths(b, (t + 1) // 2, t, rng))):
      prompt[i, :p - np_] = 0
      completion[i, nt:] = 0
    return {'do': 'score', 'rollout': _rollout(_model(case, seed), p + t), 'prompt': prompt, 'completion': completion}
  prompts = [rng.integers(3, c.vocab_size, n).astype(np.int32)
             for n in _lengths(case['prompts'], case['shortest'], case['longest'], rng)]
  sampling = {'greedy': dict(temperature=0.0, top_p=None), 'sample': dict(temperature=0.9, top_p=1.0),
              'nucleus': dict(temperature=1.0, top_p=0.95)}[case['mode']]
  config = RolloutConfig(max_tokens_to_generate=case['new'], max_prompt_length=case['longest'], seed=seed % (1 << 31),
                         kv_cache_size=case['longest'] + case['new'], eos_tokens=[-1],  # every row runs to its end
                         return_logprobs=True, **sampling)
  return {'do': 'generate', 'rollout': _rollout(_model(case, seed), config.kv_cache_size), 'config': config,
          'prompts': [p for p in prompts for _ in range(case['samples'])]}


def run(state):
  if state['do'] == 'sync':
    rollout = state['rollout']
    rollout.update_params(state['adapters'])
    return [t for layer in rollout.model().layers for key in ('qkv', 'o', 'gate_up', 'down')
            for t in (layer[key].lora_a_t, layer[key].lora_b)]
  if state['do'] == 'score':
    return state['rollout'].get_per_token_logps(state['prompt'], state['completion'])
  out = state['rollout'].generate(None, state['config'], prompt_token_ids=state['prompts'])
  return {'tokens': np.stack(out.tokens), 'logprobs': np.array(out.logprobs, dtype=np.float32)}


def _layer_weights(c, group, rank, targets, rows):
  """(bytes of one layer's matrices as a pass of `rows` rows reads them, weights a row is multiplied with)."""
  nh, kh = c.num_heads * c.head_dim, c.num_kv_heads * c.head_dim
  mats = {'q_proj': (c.embed_dim, nh), 'k_proj': (c.embed_dim, kh), 'v_proj': (c.embed_dim, kh),
          'o_proj': (nh, c.embed_dim)}
  moe = c.num_experts or 0
  if not moe:
    mats.update(gate_proj=(c.embed_dim, c.hidden_dim), up_proj=(c.embed_dim, c.hidden_dim),
                down_proj=(c.hidden_dim, c.embed_dim))
  dense = sum(k * n for k, n in mats.values())
  lora = sum(rank * sum(mats[t]) for t in targets if t in mats)
  nbytes, active = dense * (0.5 + 2.0 / group) + 2 * lora, dense + lora
  if moe:
    expert = 3 * c.embed_dim * c.hidden_dim
    touched = moe * (1.0 - (1.0 - c.num_experts_per_tok / moe) ** rows)
    nbytes += touched * expert * (0.5 + 2.0 / group) + 2 * c.embed_dim * moe
    active += c.num_experts_per_tok * expert + c.embed_dim * moe
  return nbytes, active


def work(case):
  c = _config(case)
  _, group, rank, targets = MODELS[case['model']]
  if case['do'] == 'sync':
    values = sum(t.numel() for t in _shapes(c, case['rank']))
    return {'bytes': values * (4 + 2), 'flops': 0}  # f32 in, bf16 out
  kv = c.num_layers * c.num_kv_heads * c.head_dim * 2 * 2  # bytes of a token's cache rows
  attn = 4 * c.num_layers * c.num_heads * c.head_dim       # operations of a token for each token it looks at
  head = c.vocab_size * c.embed_dim
  if case['do'] == 'score':
    rng = np.random.default_rng(0)
    b, p, t = case['sequences'], case['prompt'], case['completion']
    lens = _lengths(b, (p + 1) // 2, p, rng) + _lengths(b, (t + 1) // 2, t, rng)
    scored = int(_lengths(b, (t + 1) // 2, t, rng).sum())
    tokens = int(lens.sum())
    w, active = _layer_weights(c, group, rank, targets, tokens)
    return {'bytes': c.num_layers * w + 2 * head + 2 * tokens * kv + 8 * b * (p + t),
            'flops': 2 * tokens * c.num_layers * active + 2 * scored * head
                     + attn * float((lens.astype(float) ** 2).sum()) / 2}
  lens = np.linspace(case['longest'], case['shortest'], case['prompts']).round()
  rows, new = case['prompts'] * case['samples'], case['new']
  # the prompt once per distinct prompt, then a step per token, each of which reads every weight it uses again
  tokens = float(lens.sum())
  w, active = _layer_weights(c, group, rank, targets, tokens)
  nbytes, flops = c.num_layers * w + tokens * kv, 2 * tokens * c.num_layers * active + attn * float((lens ** 2).sum()) / 2
  w, active = _layer_weights(c, group, rank, targets, rows)
  looked_at = new * (case['samples'] * tokens + rows * new / 2)  # tokens that queries look at
  read = new * (tokens + rows * new / 2)                         # of these, rows of the cache: a prompt's once a step
  nbytes += new * (c.num_layers * w + 2 * head + rows * kv) + read * kv
  flops += new * rows * 2 * (c.num_layers * active + head) + attn * looked_at
  return {'bytes': nbytes, 'flops': flops}


def _shapes(c, rank):
  d, f, nh, kh = c.embed_dim, c.hidden_dim, c.num_heads * c.head_dim, c.num_kv_heads * c.head_dim
  for k, n in [(d, nh), (d, kh), (d, kh), (nh, d), (d, f), (d, f), (f, d)] * c.num_layers:
    yield torch.empty(k, rank, device='meta')
    yield torch.empty(rank, n, device='meta')


def tolerance(case):
  if case['do'] == 'sync':
    return 'exact'
  # Log-probs of random tokens are near -13 nats, those of greedy choices a few nats, and the logits they come from are
  # bf16: one step is 2^-5 or 2^-4 there (two batch sizes of this package differ by 0.012 and 0.002).  Tokens are the
  # same but for a near tie.
  return {'rel': 0.01} if case['do'] == 'score' else {'rel': 0.025, 'differ': 0.005}
