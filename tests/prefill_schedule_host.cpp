// Host replay of the in-place prefill schedule: the library's own planning code
// and the arithmetic its kernels share with the host, every work-group walked in
// turn.  Compiled for the host only; no kernel runs from here, so the
// registrations the compiler emits for them end in the stubs below.
#include "../k8v4-xpu_amd/csrc/prefill.hip"

#include <cstdlib>
#include <map>

extern "C" {
const char __hip_fatbin[8] = {};
void **__hipRegisterFatBinary(const void *) {
  static void *handle;
  return &handle;
}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
void __hipUnregisterFatBinary(void **) {}
}

namespace k8v4 {
namespace {
int g_cus;
std::string g_message;
}  // namespace
int device_cus() { return g_cus; }
int launch_status(const char *) { return K8V4_OK; }
void clear_error() { g_message.clear(); }
void set_error(const char *fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  std::vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_message = buf;
}

namespace {
bool fails(const char *what, int64_t x, int64_t y, int64_t z) {
  set_error("%s (%lld %lld %lld)", what, static_cast<long long>(x), static_cast<long long>(y), static_cast<long long>(z));
  return false;
}
#define CHECK(cond, x, y, z) \
  if (!(cond)) return fails(#cond, x, y, z)

bool replay_launch(const PrefillBatchArgs &ba, int head_dim, int64_t workspace_bytes) {
  const PrefillArgs &a = ba.seq[0];
  CHECK(a.total == ba.step0[ba.n], a.total, ba.step0[ba.n], 0);
  CHECK(partial_bytes(a.grid, head_dim) <= workspace_bytes, a.grid, workspace_bytes, 0);
  // Per block (numbered as for the merge): work-group -> slot, and the pages' visits.
  std::vector<std::map<int, int>> pieces(ba.block0[ba.n]);
  std::vector<std::vector<int>> visits(ba.block0[ba.n]);
  for (int i = 0; i < ba.n; ++i)
    for (int b = ba.block0[i]; b < ba.block0[i + 1]; ++b)
      visits[b].resize(block_pages(ba.seq[i], (b - ba.block0[i]) % ba.seq[i].nbh));
  for (int v = 0; v < a.grid; ++v) {
    const int s0 = range_start(a, v), s1 = range_start(a, v + 1);
    bool used[2] = {false, false};
    for (int s = s0; s < s1;) {
      int i = 0;
      while (ba.step0[i + 1] <= s) ++i;
      const PrefillArgs &sa = ba.seq[i];
      const int h = (s - ba.step0[i]) / sa.tper;
      int rb = 0, base = ba.step0[i] + h * sa.tper;
      while (rb + 1 < sa.nbh && base + block_steps(sa, rb) <= s) base += block_steps(sa, rb++);
      const int n = block_pages(sa, rb), b = ba.block0[i] + h * sa.nbh + rb;
      const auto [p_lo, p_hi, end] = piece_at(sa, base, n, s, s1);
      CHECK(h < sa.hkv && s >= base, v, i, s);
      CHECK(end > s && end <= s1, v, s, end);
      CHECK(0 <= p_lo && p_lo <= p_hi && p_hi <= n, p_lo, p_hi, n);
      s = end;
      if (p_lo == p_hi) continue;
      for (int p = p_lo; p < p_hi; ++p) ++visits[b][p];
      if (p_lo == 0 && p_hi == n) continue;
      const int slot = s0 >= base ? 0 : 1;
      CHECK(!used[slot], v, slot, b);
      used[slot] = true;
      pieces[b][v] = slot;
    }
  }
  for (int i = 0; i < ba.n; ++i) {
    const PrefillArgs &sa = ba.seq[i];
    for (int b = ba.block0[i]; b < ba.block0[i + 1]; ++b) {
      for (int c : visits[b]) CHECK(c == 1, i, b, c);
      const int h = (b - ba.block0[i]) / sa.nbh, rb = (b - ba.block0[i]) % sa.nbh;
      int start = ba.step0[i] + h * sa.tper;
      for (int r = 0; r < rb; ++r) start += block_steps(sa, r);
      int va, vb;
      page_owners(a, sa, start, block_pages(sa, rb), va, vb);
      std::map<int, int> want;
      if (va != vb)
        for (int v = va; v <= vb; ++v) want[v] = range_start(a, v) >= start ? 0 : 1;
      CHECK(pieces[b] == want, i, b, va);
    }
  }
  return true;
}
}  // namespace
}  // namespace k8v4

// 0, or 1 with the failed check in replay_message().  `in_launches`: sequences
// that share launches in place (the others run over tile images of their own).
extern "C" int replay_batch(int cus, int hkv, int head_dim, int nseq, const int64_t *q_lens, const int64_t *seq_lens,
                            int64_t workspace_bytes, int *in_launches) {
  using namespace k8v4;
  g_cus = cus;
  clear_error();
  PrefillArgs a{};
  a.hkv = hkv;
  a.rows = rows_per_block(head_dim);
  std::vector<int64_t> zeros(nseq, 0);
  BatchPlan plan;
  if (plan_batch(a, nullptr, 0, nseq, zeros.data(), q_lens, seq_lens, zeros.data(), head_dim, workspace_bytes, plan)) return 1;
  *in_launches = 0;
  for (const PrefillBatchArgs &ba : plan.launches) {
    *in_launches += ba.n;
    for (int i = 0; i < ba.n; ++i)
      if (ba.seq[i].cost != block_cost(head_dim, false)) return fails("a block's fixed cost differs in one launch", i, ba.seq[i].cost, 0), 1;
    if (!replay_launch(ba, head_dim, workspace_bytes)) return 1;
  }
  return 0;
}

extern "C" int64_t batch_workspace(int cus, int hkv, int head_dim) {
  k8v4::g_cus = cus;
  return k8v4_prefill_batch_workspace_bytes(hkv, head_dim);
}

extern "C" const char *replay_message() { return k8v4::g_message.c_str(); }
