"""Generator strategies: the native MI355X engine (replacing vLLM) and
an OpenAI-compatible HTTP client (replacing the reference's
HTTP-vLLM/argo/openai backends).

Reference parity: distllm/generate/generators/* — the `vllm` config
name is accepted as an alias of `native` so reference YAMLs keep
working; sampling defaults match vllm_backend.py:46-60 (temperature .5,
max_tokens 2000, min_p .1).
"""

from __future__ import annotations

import os
from typing import Any, Literal, Union

from pydantic import Field, model_validator

from ..registry import registry
from ..utils import BaseConfig, retry


class NativeGeneratorConfig(BaseConfig):
    """In-process generation on the native HIP engine."""

    name: Literal["native", "vllm", "huggingface"] = "native"

    @model_validator(mode="before")
    @classmethod
    def _huggingface_defaults(cls, data: Any) -> Any:
        # Drop-in acceptance of BOTH reference backend dialects:
        #  - vllm_backend.py: `llm_name` names the model
        #  - huggingface_backend.py: `pretrained_model_name_or_path`,
        #    `batch_size`, `do_sample` (False -> greedy), plus inert
        #    runtime knobs (half_precision/eval_mode/compile_model)
        #    the native engine supersedes (bf16, inference-only,
        #    hand-fused).
        if isinstance(data, dict):
            data = dict(data)  # never mutate the caller's dict
            for alias in ("llm_name", "pretrained_model_name_or_path"):
                if alias in data and "model" not in data:
                    data["model"] = data.pop(alias)
                else:
                    data.pop(alias, None)
            if "batch_size" in data:
                data.setdefault("max_batch_size",
                                data.pop("batch_size"))
            if data.pop("do_sample", True) is False:
                data.setdefault("temperature", 0.0)
            for inert in ("half_precision", "eval_mode",
                          "compile_model"):
                data.pop(inert, None)
            # Reference HuggingFaceGenerator defaults differ from
            # vLLM's: num_beams=10, top_p=.95, do_sample=True
            # (huggingface_backend.py:41-44). YAMLs naming the
            # huggingface backend and relying on defaults get those
            # semantics here too.
            if data.get("name") == "huggingface":
                data.setdefault("num_beams", 10)
                data.setdefault("top_p", 0.95)
        return data
    model: str = "llama-tiny"
    weights_path: str = ""
    tokenizer_path: str = ""
    dtype: str = "bfloat16"
    temperature: float = 0.5
    min_p: float = 0.1
    top_p: float = 0.0
    # num_beams > 1 switches to beam search (the reference's
    # huggingface backend semantics, huggingface_backend.py:41-44);
    # 0/1 = the sampling engine path
    num_beams: int = 0
    max_tokens: int = 2000
    max_batch_size: int = 64
    max_model_len: int = 4096
    # accepted for reference-YAML compatibility; single-GPU engine per
    # rank (data-parallel across ranks):
    tensor_parallel_size: int = 1
    trust_remote_code: bool = True
    # reference `quantization: true` meant NF4 capacity quantization;
    # here it opts into the CDNA4 equivalent: W8A16 fp8-e4m3 decode
    # weights (weight_dtype below)
    quantization: bool = False
    kv_cache_dtype: str = "bf16"  # or "fp8_e4m3" (CDNA4 OCP fp8)
    weight_dtype: str = "bf16"    # or "fp8_e4m3" (W8A16 decode GEMV)


class NativeGenerator:
    def __init__(self, config: NativeGeneratorConfig):
        import torch

        from ..embed.encoders import resolve_model
        from ..embed.tokenizers import load_tokenizer
        from ..engine import LLMEngine, SamplingParams
        from ..models import LayeredDims, build_model

        self.config = config
        dims, folder = resolve_model(config.model)
        device = "cuda" if torch.cuda.is_available() else "cpu"
        dtype = torch.bfloat16 if device != "cpu" else torch.float32
        if config.dtype == "float32" and isinstance(dims, LayeredDims):
            dtype = torch.float32  # their kernels run in 32-bit as well
        kw = {}
        if config.tensor_parallel_size > 1:
            import torch.distributed as dist

            if not dist.is_initialized():
                raise RuntimeError(
                    "tensor_parallel_size > 1 requires torch.distributed "
                    "(launch under torchrun with one rank per GPU)"
                )
            if dist.get_world_size() != config.tensor_parallel_size:
                raise RuntimeError(
                    "tensor_parallel_size must equal the world size "
                    "(TP subgroups are not split out)"
                )
            kw["tp_group"] = dist.group.WORLD
        self.model = build_model(dims, device=device, dtype=dtype, **kw)
        if config.weights_path or folder:
            from ..models.loader import load_weights

            load_weights(self.model, config.weights_path or folder)
        self.tokenizer = load_tokenizer(
            config.tokenizer_path or config.model,
            arch=dims.arch, vocab_size=dims.vocab_size,
            model_max_length=dims.max_position_embeddings,
        )
        wdt = config.weight_dtype
        if config.quantization and wdt == "bf16":
            if str(self.model.device).startswith("cuda"):
                wdt = "fp8_e4m3"
            else:  # reference-YAML compat field; inert off-GPU
                import warnings

                warnings.warn("quantization requested but no GPU; "
                              "keeping bf16 weights")
        self.engine = LLMEngine(self.model,
                                max_batch_size=config.max_batch_size,
                                max_model_len=config.max_model_len,
                                kv_cache_dtype=config.kv_cache_dtype,
                                weight_dtype=wdt)
        # vLLM-style capture-at-init: pre-record every pow2 decode
        # graph bucket so batch drain never captures inside a timed /
        # serving window (measured ~0.2s per first-use capture)
        if self.engine.use_graphs:
            b, buckets = 1, []
            while b < config.max_batch_size:
                buckets.append(b)
                b <<= 1
            buckets.append(config.max_batch_size)
            self.engine.warm_graphs(sorted(set(buckets)))
        self._loop = None
        eos = getattr(self.tokenizer, "eos_token_id", None)
        self.params = SamplingParams(
            temperature=config.temperature,
            min_p=config.min_p,
            top_p=config.top_p if config.top_p > 0 else 1.0,
            max_tokens=config.max_tokens,
            stop_token_ids=(eos,) if eos is not None else (),
        )

    def get_loop(self):
        """Online engine loop (request-level continuous batching);
        once created it owns the engine and all generate() calls route
        through it (thread-safe)."""
        if self._loop is None:
            from ..engine.loop import EngineLoop

            self._loop = EngineLoop(self.engine, self.params)
        return self._loop

    def generate_one(self, prompt: str) -> str:
        loop = self.get_loop()
        ids = self._tokenize([prompt])[0]
        out = loop.generate([ids])[0]
        return self.tokenizer.decode(out, skip_special_tokens=True)

    def _tokenize(self, prompts: list[str]) -> list[list[int]]:
        enc = self.tokenizer(prompts, padding=False, truncation=True,
                             return_tensors=None)
        ids = enc["input_ids"]
        import torch

        if isinstance(ids, torch.Tensor):
            mask = enc["attention_mask"]
            return [ids[i][mask[i].bool()].tolist()
                    for i in range(len(prompts))]
        return [list(x) for x in ids]

    def generate(self, prompts: list[str]) -> list[str]:
        if isinstance(prompts, str):
            prompts = [prompts]
        prompt_ids = self._tokenize(prompts)
        if self.config.num_beams and self.config.num_beams > 1:
            from ..engine.beam import beam_generate

            eos = getattr(self.tokenizer, "eos_token_id", None)
            out_ids = [
                beam_generate(self.engine.model, p,
                              self.config.num_beams,
                              self.params.max_tokens, eos_token_id=eos)
                for p in prompt_ids
            ]
        elif self._loop is not None:  # loop owns the engine once started
            out_ids = self._loop.generate(prompt_ids)
        else:
            out_ids = self.engine.generate(prompt_ids, self.params)
        return [
            self.tokenizer.decode(o, skip_special_tokens=True)
            for o in out_ids
        ]


class OpenAICompatGeneratorConfig(BaseConfig):
    """HTTP client against any OpenAI-compatible /v1 server (our
    chat_server, a remote endpoint, or an Argo-style proxy)."""

    name: Literal["openai_http", "argo"] = "openai_http"
    base_url: str = "http://localhost:8000/v1"
    model: str = "default"
    api_key_env: str = Field(
        "OPENAI_API_KEY", description="env var holding the key, if any"
    )
    api_key: str = Field(
        "", description="literal key (reference argoproxy-style configs "
        "pass the key inline; takes precedence over api_key_env)"
    )
    temperature: float = 0.5
    max_tokens: int = 2000
    timeout: float = 120.0
    use_chat_endpoint: bool = True


class OpenAICompatGenerator:
    def __init__(self, config: OpenAICompatGeneratorConfig):
        import httpx

        self.config = config
        headers = {}
        key = config.api_key or os.environ.get(config.api_key_env, "")
        if key:
            headers["Authorization"] = f"Bearer {key}"
        self._client = httpx.Client(base_url=config.base_url,
                                    headers=headers,
                                    timeout=config.timeout)

    @retry(tries=5, base_delay=1.0)
    def _one(self, prompt: str) -> str:
        c = self.config
        if c.use_chat_endpoint:
            r = self._client.post("/chat/completions", json={
                "model": c.model,
                "messages": [{"role": "user", "content": prompt}],
                "temperature": c.temperature,
                "max_tokens": c.max_tokens,
            })
            r.raise_for_status()
            return r.json()["choices"][0]["message"]["content"]
        r = self._client.post("/completions", json={
            "model": c.model, "prompt": prompt,
            "temperature": c.temperature, "max_tokens": c.max_tokens,
        })
        r.raise_for_status()
        return r.json()["choices"][0]["text"]

    def generate(self, prompts: list[str]) -> list[str]:
        if isinstance(prompts, str):
            prompts = [prompts]
        return [self._one(p) for p in prompts]


GeneratorConfigs = Union[NativeGeneratorConfig, OpenAICompatGeneratorConfig]



class ApiGeneratorConfig(BaseConfig):
    """API-model generation (reference `langchain` backend parity:
    distllm/generate/generators/langchain_backend.py — gpt-3.5-turbo /
    gemini-pro / claude-3-opus via API keys in a .env file). SDK-free:
    the three wire protocols are spoken directly over httpx."""

    name: Literal["langchain", "api"] = "langchain"
    llm: str = Field("gpt-3.5-turbo",
                     description="gpt-* | gemini-* | claude-* model id")
    temperature: float = 0.0
    max_tokens: int = 2000
    verbose: bool = True
    dotenv_path: str = "~/.env"
    timeout: float = 120.0


class ApiGenerator:
    """Dispatches on the model-id prefix to the OpenAI, Google
    Generative Language or Anthropic Messages REST APIs."""

    def __init__(self, config: ApiGeneratorConfig):
        self.config = config
        self._load_dotenv(config.dotenv_path)

    @staticmethod
    def _load_dotenv(path: str) -> None:
        """Minimal .env loader (python-dotenv-free): KEY=VALUE lines,
        existing environment wins (reference load_dotenv semantics)."""
        import pathlib

        p = pathlib.Path(path).expanduser()
        if not p.exists():
            return
        for line in p.read_text().splitlines():
            line = line.strip()
            if not line or line.startswith("#") or "=" not in line:
                continue
            k, _, v = line.partition("=")
            os.environ.setdefault(k.strip(), v.strip().strip("'\""))

    def build_request(self, prompt: str):
        """(url, headers, json_body, parse) for one prompt — separated
        from the HTTP send so the wire formats are unit-testable
        offline."""
        c = self.config
        m = c.llm
        if m.startswith("gemini"):
            key = os.environ.get("GOOGLE_API_KEY", "")
            url = ("https://generativelanguage.googleapis.com/v1beta/"
                   f"models/{m}:generateContent?key={key}")
            body = {
                "contents": [{"parts": [{"text": prompt}]}],
                "generationConfig": {"temperature": c.temperature,
                                     "maxOutputTokens": c.max_tokens},
            }

            def parse(j):
                return j["candidates"][0]["content"]["parts"][0]["text"]

            return url, {"Content-Type": "application/json"}, body, parse
        if m.startswith("claude"):
            url = "https://api.anthropic.com/v1/messages"
            headers = {
                "x-api-key": os.environ.get("ANTHROPIC_API_KEY", ""),
                "anthropic-version": "2023-06-01",
                "Content-Type": "application/json",
            }
            body = {
                "model": m,
                "max_tokens": c.max_tokens,
                "temperature": c.temperature,
                "messages": [{"role": "user", "content": prompt}],
            }

            def parse(j):
                return j["content"][0]["text"]

            return url, headers, body, parse
        # default: OpenAI chat completions (gpt-*)
        url = "https://api.openai.com/v1/chat/completions"
        headers = {
            "Authorization":
                f"Bearer {os.environ.get('OPENAI_API_KEY', '')}",
            "Content-Type": "application/json",
        }
        body = {
            "model": m,
            "temperature": c.temperature,
            "max_tokens": c.max_tokens,
            "messages": [{"role": "user", "content": prompt}],
        }

        def parse(j):
            return j["choices"][0]["message"]["content"]

        return url, headers, body, parse

    @retry(tries=3, base_delay=1.0)
    def _send(self, url, headers, body, parse) -> str:
        import httpx

        r = httpx.post(url, headers=headers, json=body,
                       timeout=self.config.timeout)
        r.raise_for_status()
        return parse(r.json())

    def generate(self, prompts):
        if isinstance(prompts, str):
            prompts = [prompts]
        out = []
        for p in prompts:
            out.append(self._send(*self.build_request(p)))
        return out


STRATEGIES: dict[str, tuple[type, type]] = {
    "native": (NativeGeneratorConfig, NativeGenerator),
    "vllm": (NativeGeneratorConfig, NativeGenerator),
    "huggingface": (NativeGeneratorConfig, NativeGenerator),
    "openai_http": (OpenAICompatGeneratorConfig, OpenAICompatGenerator),
    "argo": (OpenAICompatGeneratorConfig, OpenAICompatGenerator),
    "langchain": (ApiGeneratorConfig, ApiGenerator),
    "api": (ApiGeneratorConfig, ApiGenerator),
}


def _factory(kwargs: dict[str, Any]):
    name = kwargs.get("name", "")
    if name not in STRATEGIES:
        raise ValueError(
            f"unknown generator name {name!r}; options: {sorted(STRATEGIES)}"
        )
    cfg_cls, impl_cls = STRATEGIES[name]
    return impl_cls(cfg_cls(**kwargs))


def get_generator(kwargs: dict[str, Any], register: bool = False):
    if register:
        return registry.get(_factory, dict(kwargs))
    return _factory(dict(kwargs))
