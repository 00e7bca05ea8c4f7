// oxs_dfa.hip — grammar masks from a DFA for MI355X (gfx950).
//
// For a batch of rows, each in its own DFA state, walks every vocabulary
// token's bytes through the transition table (crates/oxide-core/src/dfa.rs:110-148,
// crates/oxide-server/src/grammar_engine.rs:42-65) and writes the packed
// allowed-token bitmask that oxs_sample_batch reads (oxs_batch.allowed_mask).
//
// One thread per token. Its bytes come in 16-byte pieces, and each piece is
// walked from up to 64 start states (every state of a small table, or the
// states of 64 rows): a table of the start states that accept each first byte
// leaves few walks, and tables of up to 8 states compose whole transition
// functions with byte permutes. The tokens' results are turned into one mask
// word per start state and 32 tokens, which the rows then copy. Bound: latency
// (the token bytes and offsets are read once per row group; the masks are
// written once).
//
// A walk depends only on the state it starts from, so a decode loop computes
// the masks of every state once per grammar and vocabulary (this kernel over
// the states themselves) and gathers one row per sequence each step
// (mask_gather_kernel): a copy of ceil(V / 32) words per row.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/oxide_sampler.h"

namespace oxs_grammar {

constexpr int kThreads = 256;
constexpr int kTok = 2;               // tokens per thread
constexpr int kWords = kTok * kThreads / 32;  // mask words per row and block
constexpr int kRows = 128;            // rows per block with a walk from every state
constexpr uint32_t kList = 64;        // start states walked together
constexpr int kIlp = 4;               // of them, by one thread at the same time
constexpr uint32_t kPermStates = 8;   // tables whose transition functions fit a byte permute
constexpr uint32_t kLdsStates = 128;  // tables of up to 128 states are kept in LDS, a byte per entry
constexpr uint32_t kErr = OXS_DFA_ERROR_STATE;

struct Params {
  const uint32_t* trans;
  uint32_t num_states;
  const uint32_t* offsets;
  const uint8_t* bytes;
  uint32_t num_bytes;
  uint32_t V;
  const uint32_t* states;
  uint32_t B;
  uint32_t* mask;
  int64_t mask_ld;
};

// Next states as bytes. With kPermStates states a byte is also a v_perm_b32
// selector: 0-7 pick a byte of the function, anything from 0x0d up gives 0xff.
// So a walk that left the table (kOut: allowed if its token ends there) or
// failed (kDead) fails at its next byte by itself. Larger tables use the same
// two marks above their states.
constexpr uint32_t kDead = 0xffu;
__device__ __forceinline__ uint32_t next_byte(uint32_t next, uint32_t ns, uint32_t out) {
  return next == kErr ? kDead : next < ns ? next : out;
}

// How a block walks: kPerm8 every state of a table of up to 8, by composing
// byte functions; kLds and kGlobal a list of up to 64 start states, one walk
// per start state that accepts the token's first byte, through the table's
// bytes in LDS or its words in memory.
enum Walk { kPerm8, kLds, kGlobal };

// Bytes [at, at + 16) of the token bytes, zeros past num_bytes. (Unaligned
// 16-byte loads are one instruction.)
struct __attribute__((packed)) Piece {
  uint32_t w[4];
};
__device__ __forceinline__ void load_piece(const Params& p, uint32_t at, uint32_t (&w)[4]) {
  if (p.num_bytes - at >= 16u) {  // (at <= num_bytes)
    const Piece q = *(const Piece*)(p.bytes + at);
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = q.w[i];
  } else {
    uint64_t lo = 0, hi = 0;
    for (uint32_t i = p.num_bytes - at; i-- > 0u;) {  // (at most 15)
      hi = (hi << 8) | (lo >> 56);
      lo = (lo << 8) | p.bytes[at + i];
    }
    w[0] = (uint32_t)lo;
    w[1] = (uint32_t)(lo >> 32);
    w[2] = (uint32_t)hi;
    w[3] = (uint32_t)(hi >> 32);
  }
}

// Masks of kTok * 256 tokens for a group of rows. by_state: the start states
// are the table's own (num_states <= 64) and blockIdx.y picks kRows rows;
// otherwise they are the states of the 64 rows that blockIdx.y picks.
//
// Measured, us per launch, in brackets with one walk after the other per thread:
// 128 rows x 128256 tokens, a fixed-prefix grammar (few start states accept a first
// byte) of 8 states 7.7 (walks nothing), 16 states 13.0 (17.6), 64 states 25.7 (32.9), 129
// states 22.9 (28.3); tables without error entries of 16 states 24.9 (57.5), 300
// states 208 (376). One row, 64 states 8.4 (8.3).
template <Walk WALK>
__global__ __launch_bounds__(kThreads) void dfa_mask_kernel(const Params p, const uint32_t by_state) {
  extern __shared__ __align__(16) uint8_t s_table[];  // kLds: [num_states][256] next states
  __shared__ uint64_t s_fn[256];  // kPerm8: byte b's function; else: the start states that accept b
  __shared__ uint32_t s_start[kList];
  __shared__ uint32_t s_words[kList + 1][kWords];  // [start state][word]; the last: tokens with no bytes
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t ns = p.num_states;
  const uint32_t out = WALK == kPerm8 ? 0x0du : 0xfeu;  // (kLds: num_states <= 128 < 0xfe)
  const uint32_t words = (p.V + 31u) / 32u;
  const uint32_t tbase = blockIdx.x * (kTok * kThreads);
  const uint32_t r0 = blockIdx.y * (by_state ? (uint32_t)kRows : kList);
  const uint32_t nr = min(by_state ? (uint32_t)kRows : kList, p.B - r0);
  const uint32_t n_list = by_state ? ns : nr;

  uint32_t b0[kTok], len[kTok], piece[kTok][4];
  bool in[kTok];
#pragma unroll
  for (int k = 0; k < kTok; ++k) {
    const uint32_t t = tbase + k * kThreads + tid;
    in[k] = t < p.V;
    const uint32_t at = in[k] ? t : 0u;
    b0[k] = p.offsets[at];
    const uint32_t e = p.offsets[at + 1];
    if (e < b0[k] || e > p.num_bytes) in[k] = false;  // a range outside the byte array: not allowed, nothing read
    len[k] = in[k] ? e - b0[k] : 0u;
    if (!in[k]) b0[k] = 0u;
  }
  if (WALK != kPerm8) {
    if (tid < kList) s_start[tid] = by_state ? tid : p.states[r0 + min(tid, nr - 1u)];
    if (WALK == kLds)
      for (uint32_t i = tid; i < ns * 64u; i += kThreads) {  // four entries per step
        const uint32_t* q = p.trans + 4u * i;
        uint32_t w = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) w |= next_byte(q[e], ns, out) << (8 * e);
        ((uint32_t*)s_table)[i] = w;
      }
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < kTok; ++k)
    if (len[k]) load_piece(p, b0[k], piece[k]);
  {  // this thread's byte: its function, or the start states that accept it
    uint64_t f = 0;
    if constexpr (WALK == kPerm8) {
      uint32_t nx[kPermStates];
#pragma unroll
      for (uint32_t s = 0; s < kPermStates; ++s) nx[s] = kErr;
      if (ns) {
#pragma unroll
        for (uint32_t s = 0; s < kPermStates; ++s) nx[s] = p.trans[(s < ns ? s : 0u) * 256u + tid];
      }
#pragma unroll
      for (uint32_t s = 0; s < kPermStates; ++s)
        f |= (uint64_t)(s < ns ? next_byte(nx[s], ns, out) : kDead) << (8u * s);
    } else {
      for (uint32_t i0 = 0; i0 < n_list; i0 += 8u) {  // eight reads at a time
        uint32_t nx[8], st[8];
#pragma unroll
        for (uint32_t e = 0; e < 8; ++e) {
          st[e] = s_start[min(i0 + e, n_list - 1u)];
          const uint32_t at = (st[e] < ns ? st[e] : 0u);
          nx[e] = WALK == kLds ? (s_table[at * 256u + tid] == kDead ? kErr : 0u) : p.trans[(size_t)at * 256u + tid];
        }
#pragma unroll
        for (uint32_t e = 0; e < 8; ++e)
          if (i0 + e < n_list && st[e] < ns && nx[e] != kErr) f |= 1ull << (i0 + e);
      }
    }
    s_fn[tid] = f;
  }
  __syncthreads();

#pragma unroll
  for (int k = 0; k < kTok; ++k) {
    uint64_t alive = 0;  // bit i: the token walks from start state i
    if constexpr (WALK == kPerm8) {
      uint32_t lo = 0x03020100u, hi = 0x07060504u;  // the states reached, one byte each
      for (uint32_t j0 = 0; j0 < len[k]; j0 += 16u) {
        if (j0) load_piece(p, b0[k] + j0, piece[k]);
        const uint32_t n = min(len[k] - j0, 16u);
#pragma unroll
        for (uint32_t j = 0; j < 16; ++j) {
          if (j < n) {
            const uint64_t f = s_fn[(piece[k][j / 4] >> (8u * (j % 4u))) & 0xffu];
            lo = __builtin_amdgcn_perm((uint32_t)(f >> 32), (uint32_t)f, lo);
            hi = __builtin_amdgcn_perm((uint32_t)(f >> 32), (uint32_t)f, hi);
          }
        }
      }
      // (bytes below 0x80: a state, or kOut)
#pragma unroll
      for (uint32_t s = 0; s < kPermStates; ++s)
        alive |= (uint64_t)((~(s < 4u ? lo : hi) >> (8u * (s % 4u) + 7u)) & 1u) << s;
      alive &= (1ull << ns) - 1ull;
    } else if (len[k] == 0u) {
      alive = ~0ull;
    } else {
      uint64_t todo = s_fn[piece[k][0] & 0xffu];
      if (len[k] == 1u) {
        alive = todo;
      } else {
        // the start states that accept the first byte. A walk is a chain of
        // dependent reads, so kIlp of them are kept in flight while any token of the
        // wavefront has more than one left.
        constexpr uint32_t dead = WALK == kLds ? kDead : kErr;
        const auto walk = [&](auto ilp) {
          constexpr int ILP = decltype(ilp)::value;
          uint32_t c[ILP];
          uint64_t bit[ILP];
#pragma unroll
          for (int e = 0; e < ILP; ++e) {
            bit[e] = todo & (0ull - todo);
            c[e] = todo ? s_start[__builtin_ctzll(todo)] : dead;
            todo &= todo - 1ull;
          }
          for (uint32_t j0 = 0; j0 < len[k]; j0 += 16u) {
            uint32_t w[4] = {piece[k][0], piece[k][1], piece[k][2], piece[k][3]};
            if (j0) load_piece(p, b0[k] + j0, w);
            const uint32_t n = min(len[k] - j0, 16u);
            bool any = true;
#pragma unroll
            for (uint32_t j = 0; j < 16; ++j) {
              if (j < n && any) {  // (DfaSchemaGrammar::transition, dfa.rs:110-126)
                const uint32_t b = (w[j / 4] >> (8u * (j % 4u))) & 0xffu;
                uint32_t nx[ILP];
#pragma unroll
                for (int e = 0; e < ILP; ++e) {
                  const uint32_t at = c[e] < ns ? c[e] : 0u;
                  nx[e] = WALK == kLds ? s_table[at * 256u + b] : p.trans[(size_t)at * 256u + b];
                }
                uint32_t all = dead;
#pragma unroll
                for (int e = 0; e < ILP; ++e) {
                  c[e] = c[e] < ns ? nx[e] : dead;  // (a walk outside the table fails at its next byte)
                  all &= c[e];
                }
                any = all != dead;
              }
            }
            if (!any) break;
          }
#pragma unroll
          for (int e = 0; e < ILP; ++e) alive |= c[e] != dead ? bit[e] : 0ull;
        };
        while (__any((todo & (todo - 1ull)) != 0ull)) walk(std::integral_constant<int, kIlp>{});
        if (todo) walk(std::integral_constant<int, 1>{});
      }
    }
    if (!in[k]) alive = 0;
    // lane i takes the ballot of start state i
    const uint32_t w = (k * kThreads + 64u * wave) / 32u;
    uint32_t mine_lo = 0, mine_hi = 0;
    for (uint32_t i = 0; i < n_list; ++i) {
      const uint64_t m = __ballot((alive >> i) & 1ull);
      mine_lo = lane == i ? (uint32_t)m : mine_lo;
      mine_hi = lane == i ? (uint32_t)(m >> 32) : mine_hi;
    }
    if (lane < n_list) {
      s_words[lane][w] = mine_lo;
      s_words[lane][w + 1] = mine_hi;
    }
    const uint64_t empty = __ballot(in[k] && len[k] == 0u);  // allowed from every state, even outside the table
    if (lane == 0) {
      s_words[kList][w] = (uint32_t)empty;
      s_words[kList][w + 1] = (uint32_t)(empty >> 32);
    }
  }
  __syncthreads();
  for (uint32_t i = tid; i < nr * (uint32_t)kWords; i += kThreads) {
    const uint32_t q = i / kWords, w = i % kWords;
    const uint32_t gw = blockIdx.x * kWords + w;
    uint32_t idx = q;
    if (by_state) {
      const uint32_t s = p.states[r0 + q];
      idx = s < ns ? s : kList;
    }
    if (gw < words) p.mask[(size_t)(r0 + q) * p.mask_ld + gw] = s_words[idx][w];
  }
}

// Row b of the output is row min(states[b], num_states) of the per-state
// masks (row num_states holds the masks of every state outside the table).
constexpr int kGatherWords = 4 * kThreads;  // words per gather block
__global__ __launch_bounds__(kThreads) void mask_gather_kernel(const uint32_t* __restrict__ table, uint32_t num_states,
                                                              int64_t table_ld, uint32_t words,
                                                              const uint32_t* __restrict__ states,
                                                              uint32_t* __restrict__ mask, int64_t mask_ld) {
  const uint32_t row = blockIdx.y;
  const uint32_t s = min(states[row], num_states);
  const uint32_t* src = table + (size_t)s * table_ld;
  uint32_t* dst = mask + (size_t)row * mask_ld;
  const uint32_t w0 = blockIdx.x * kGatherWords;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t w = w0 + k * kThreads + threadIdx.x;
    if (w < words) dst[w] = src[w];
  }
}

// ---------------------------------------------------------------- static masks

// The first character of a token's text, decoded from UTF-8 (Rust's
// text.chars().next()); a malformed sequence (bad continuation, truncation,
// overlong form, surrogate, beyond U+10FFFF) gives U+FFFD, as a lossy decode
// would (the reference's vocabulary is always valid UTF-8).
__device__ __forceinline__ uint32_t first_char(const uint8_t* b, uint32_t len) {
  const uint32_t c0 = b[0];
  if (c0 < 0x80u) return c0;
  uint32_t n, c;
  if ((c0 & 0xe0u) == 0xc0u) { n = 1; c = c0 & 0x1fu; }
  else if ((c0 & 0xf0u) == 0xe0u) { n = 2; c = c0 & 0x0fu; }
  else if ((c0 & 0xf8u) == 0xf0u) { n = 3; c = c0 & 0x07u; }
  else return 0xfffdu;
  if (len < n + 1) return 0xfffdu;
  for (uint32_t i = 1; i <= n; ++i) {
    const uint32_t ci = b[i];
    if ((ci & 0xc0u) != 0x80u) return 0xfffdu;
    c = (c << 6) | (ci & 0x3fu);
  }
  const uint32_t least = n == 1 ? 0x80u : n == 2 ? 0x800u : 0x10000u;
  if (c < least || (c >= 0xd800u && c <= 0xdfffu) || c > 0x10ffffu) return 0xfffdu;
  return c;
}

__device__ __forceinline__ void write_mask_bits(bool ok, uint32_t t, uint32_t words, uint32_t* mask) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint64_t m = __ballot(ok);
  const uint32_t wbase = (t - lane) / 32u;
  if (lane == 0 && wbase < words) mask[wbase] = (uint32_t)m;
  if (lane == 32 && wbase + 1 < words) mask[wbase + 1] = (uint32_t)(m >> 32);
}

struct GbnfParams {
  const uint32_t* ranges;  // [n_ranges][2]
  uint32_t n_ranges;
  const uint32_t* lit_off;  // [n_lits + 1]
  const uint8_t* lit_bytes;
  uint32_t n_lits;
  const uint32_t* offsets;
  const uint8_t* bytes;
  uint32_t num_bytes;
  uint32_t V;
  uint32_t* mask;
};

// GbnfGrammarEngine::apply_grammar_mask (crates/oxide-core/src/sampler.rs:555-583):
// a token with no characters is left alone; otherwise it is allowed when its
// first character lies in one of the rule's ranges, or when a literal starts
// with its text or its text starts with a literal. One thread per token.
__global__ __launch_bounds__(kThreads) void gbnf_mask_kernel(const GbnfParams p) {
  const uint32_t t = blockIdx.x * kThreads + threadIdx.x;
  bool ok = false;
  if (t < p.V) {
    const uint32_t b0 = p.offsets[t], e = p.offsets[t + 1];
    if (e >= b0 && e <= p.num_bytes) {
      const uint32_t len = e - b0;
      const uint8_t* tb = p.bytes + b0;
      if (len == 0) {
        ok = true;  // text.chars().next() is None: not masked
      } else {
        const uint32_t c = first_char(tb, len);
        for (uint32_t i = 0; i < p.n_ranges && !ok; ++i) ok = c >= p.ranges[2 * i] && c <= p.ranges[2 * i + 1];
        for (uint32_t i = 0; i < p.n_lits && !ok; ++i) {
          const uint32_t lb = p.lit_off[i], ll = p.lit_off[i + 1] - lb;
          const uint32_t n = min(ll, len);  // lit.starts_with(text) || text.starts_with(lit): equal first n bytes
          bool same = true;
          for (uint32_t j = 0; j < n && same; ++j) same = p.lit_bytes[lb + j] == tb[j];
          ok = same;
        }
      }
    }
  }
  write_mask_bits(ok, t, (p.V + 31u) / 32u, p.mask);
}

// GrammarLogitMasker::mask_logits (crates/oxide-core/src/grammar_mask.rs:55-65):
// a token whose byte b is given (token_ascii[t] < 256) is masked unless
// allowed[b]; a token without one (Rust's None) is left alone.
__global__ __launch_bounds__(kThreads) void ascii_mask_kernel(const uint8_t* __restrict__ allowed,
                                                             const uint16_t* __restrict__ token_ascii, uint32_t V,
                                                             uint32_t* __restrict__ mask) {
  const uint32_t t = blockIdx.x * kThreads + threadIdx.x;
  bool ok = false;
  if (t < V) {
    const uint32_t b = token_ascii[t];
    ok = b >= 256u || allowed[b] != 0;
  }
  write_mask_bits(ok, t, (V + 31u) / 32u, mask);
}

}  // namespace oxs_grammar

extern "C" int oxs_dfa_mask(const oxs_dfa* dfa, const oxs_token_bytes* tokens, const uint32_t* states,
                            uint32_t batch, uint32_t* mask, int64_t mask_ld, void* stream) {
  using namespace oxs_grammar;
  if (!dfa || !tokens) return OXS_ERR_INVALID_ARGUMENT;
  if (batch == 0 || tokens->vocab == 0) return OXS_OK;
  if ((dfa->num_states && !dfa->transitions) || !tokens->offsets || !tokens->bytes || !states || !mask)
    return OXS_ERR_INVALID_ARGUMENT;
  if (mask_ld < (int64_t)((tokens->vocab + 31u) / 32u)) return OXS_ERR_INVALID_ARGUMENT;
  // token indices stay below 2^31; at most 65535 x 16 rows, within the grid's y extent
  // (a block covers 64 or 128)
  if (tokens->vocab > (1u << 31) || batch > 65535u * 16u) return OXS_ERR_INVALID_ARGUMENT;
  Params p;
  p.trans = dfa->transitions;
  p.num_states = dfa->num_states;
  p.offsets = tokens->offsets;
  p.bytes = tokens->bytes;
  p.num_bytes = tokens->num_bytes;
  p.V = tokens->vocab;
  p.states = states;
  p.B = batch;
  p.mask = mask;
  p.mask_ld = mask_ld;
  hipStream_t st = (hipStream_t)stream;
  const uint32_t ns = p.num_states;
  // start states: the table's own when there are at most 64 and the rows are no
  // fewer (or there are at most 8, which are walked at once), else the rows'
  const uint32_t by_state = ns <= kPermStates || (ns <= kList && batch > ns) ? 1u : 0u;
  const uint32_t per_block = (uint32_t)(kTok * kThreads), rows = by_state ? (uint32_t)kRows : kList;
  const dim3 grid((p.V + per_block - 1) / per_block, (batch + rows - 1) / rows);
  if (ns <= kPermStates) hipLaunchKernelGGL(dfa_mask_kernel<kPerm8>, grid, dim3(kThreads), 0, st, p, by_state);
  else if (ns <= kLdsStates)
    hipLaunchKernelGGL(dfa_mask_kernel<kLds>, grid, dim3(kThreads), ns * 256u, st, p, by_state);
  else hipLaunchKernelGGL(dfa_mask_kernel<kGlobal>, grid, dim3(kThreads), 0, st, p, by_state);
  return hipGetLastError() == hipSuccess ? OXS_OK : OXS_ERR_HIP;
}

extern "C" int oxs_dfa_mask_gather(const uint32_t* state_masks, uint32_t num_states, int64_t state_masks_ld,
                                   uint32_t vocab, const uint32_t* states, uint32_t batch, uint32_t* mask,
                                   int64_t mask_ld, void* stream) {
  using namespace oxs_grammar;
  if (batch == 0 || vocab == 0) return OXS_OK;
  const uint32_t words = (vocab + 31u) / 32u;
  if (!state_masks || !states || !mask || state_masks_ld < (int64_t)words || mask_ld < (int64_t)words)
    return OXS_ERR_INVALID_ARGUMENT;
  if (batch > 65535u) return OXS_ERR_INVALID_ARGUMENT;  // one grid row per batch row
  const dim3 grid((words + kGatherWords - 1) / kGatherWords, batch);
  hipLaunchKernelGGL(mask_gather_kernel, grid, dim3(kThreads), 0, (hipStream_t)stream, state_masks, num_states,
                     state_masks_ld, words, states, mask, mask_ld);
  return hipGetLastError() == hipSuccess ? OXS_OK : OXS_ERR_HIP;
}

extern "C" int oxs_gbnf_mask(const oxs_gbnf_rule* rule, const oxs_token_bytes* tokens, uint32_t* mask,
                             void* stream) {
  using namespace oxs_grammar;
  if (!rule || !tokens) return OXS_ERR_INVALID_ARGUMENT;
  if (tokens->vocab == 0) return OXS_OK;
  if (!tokens->offsets || !tokens->bytes || !mask || (rule->num_ranges && !rule->ranges) ||
      (rule->num_literals && (!rule->literal_offsets || !rule->literal_bytes)))
    return OXS_ERR_INVALID_ARGUMENT;
  if (tokens->vocab > (1u << 31)) return OXS_ERR_INVALID_ARGUMENT;
  GbnfParams p;
  p.ranges = rule->ranges;
  p.n_ranges = rule->num_ranges;
  p.lit_off = rule->literal_offsets;
  p.lit_bytes = rule->literal_bytes;
  p.n_lits = rule->num_literals;
  p.offsets = tokens->offsets;
  p.bytes = tokens->bytes;
  p.num_bytes = tokens->num_bytes;
  p.V = tokens->vocab;
  p.mask = mask;
  hipLaunchKernelGGL(gbnf_mask_kernel, dim3((p.V + kThreads - 1) / kThreads), dim3(kThreads), 0,
                     (hipStream_t)stream, p);
  return hipGetLastError() == hipSuccess ? OXS_OK : OXS_ERR_HIP;
}

extern "C" int oxs_ascii_mask(const uint8_t* allowed_ascii, const uint16_t* token_ascii, uint32_t vocab,
                              uint32_t* mask, void* stream) {
  using namespace oxs_grammar;
  if (vocab == 0) return OXS_OK;
  if (!allowed_ascii || !token_ascii || !mask || vocab > (1u << 31)) return OXS_ERR_INVALID_ARGUMENT;
  hipLaunchKernelGGL(ascii_mask_kernel, dim3((vocab + kThreads - 1) / kThreads), dim3(kThreads), 0,
                     (hipStream_t)stream, allowed_ascii, token_ascii, vocab, mask);
  return hipGetLastError() == hipSuccess ? OXS_OK : OXS_ERR_HIP;
}
