// The resident kernels' transforms (spk_line_fft.hpp) on the CPU: a host thread
// for each thread of a workgroup, __syncthreads a barrier over all of them and
// wave_lds_order one over a wavefront's 64.  LDS and the twiddle table are
// exactly sized heap arrays, so that a sanitizer build reports a slot out of
// range; values are compared with a direct FP64 transform.  Also the positions
// of the four-column column pass against the layouts' own.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <pthread.h>
#include <thread>
#include <vector>

#define __device__
#define __forceinline__ inline
static thread_local struct { int x; } threadIdx;
static pthread_barrier_t g_all;
static std::vector<pthread_barrier_t> g_wave;
static void __syncthreads() { pthread_barrier_wait(&g_all); }

#include "spk_line_fft.hpp"

namespace spk {
void wave_lds_order() { pthread_barrier_wait(&g_wave[threadIdx.x / 64]); }
}  // namespace spk
using namespace spk;

namespace {

double error(const std::vector<c32>& got, const std::vector<double>& re,
             const std::vector<double>& im) {
  double num = 0, den = 0;
  for (size_t i = 0; i < got.size(); ++i) {
    num += (got[i].x - re[i]) * (got[i].x - re[i]) + (got[i].y - im[i]) * (got[i].y - im[i]);
    den += re[i] * re[i] + im[i] * im[i];
  }
  return std::sqrt(num / den);
}

template <int N, int TT, bool LEAN>
int check() {
  using LF = LineFft<N, TT, LEAN>;
  constexpr int E = 8, T = N / E, NT = T * TT;
  std::vector<c32> table(N, c32{0.0f, 0.0f}), in(N * TT);
  auto w = [](int m) {
    const double a = -2.0 * M_PI * m / N;
    return c32{(float)std::cos(a), (float)std::sin(a)};
  };
  for (int s = 1; s < plan_stages(N, E); ++s) {
    const int R = plan_radix(N, E, s), off = staged_tw_offset(N, E, s);
    int ns = 1;
    for (int i = 0; i < s; ++i) ns *= plan_radix(N, E, i);
    for (int k = 0; k < ns; ++k)
      for (int r = 1; r < R; ++r)
        table[off + k * (R - 1) + r - 1] = w(staged_tw_exponent(N, E, s, k, r));
  }
  for (size_t i = 0; i < in.size(); ++i)
    in[i] = c32{(float)((i * 2654435761u) % 1000) * 1e-3f - 0.5f,
                (float)((i * 40503u + 7) % 997) * 1e-3f - 0.5f};
  std::vector<double> re(N * TT), im(N * TT), sre(N * TT), sim(N * TT);
  for (int b = 0; b < TT; ++b)
    for (int k = 0; k < N; ++k) {
      double x = 0, y = 0;
      for (int j = 0; j < N; ++j) {
        const double a = -2.0 * M_PI * (int)((long long)j * k % N) / N;
        const c32 v = in[b * N + j];
        x += v.x * std::cos(a) - v.y * std::sin(a);
        y += v.x * std::sin(a) + v.y * std::cos(a);
      }
      re[b * N + k] = x;
      im[b * N + k] = y;
      sre[b * N + k] = (double)N * in[b * N + k].x;
      sim[b * N + k] = (double)N * in[b * N + k].y;
    }
  // forward, forward and back, forward and moved
  std::vector<c32> lds(LF::LDS), fwd(N * TT), back(N * TT), moved(N * TT);
  std::vector<int> hooks(NT, 0);
  pthread_barrier_init(&g_all, nullptr, NT);
  g_wave.resize((NT + 63) / 64);
  for (size_t i = 0; i < g_wave.size(); ++i)
    pthread_barrier_init(&g_wave[i], nullptr, std::min(64, NT - 64 * (int)i));
  std::vector<std::thread> threads;
  for (int tid = 0; tid < NT; ++tid)
    threads.emplace_back([&, tid]() {
      threadIdx.x = tid;
      LF tf;
      tf.init(lds.data(), table.data());
      auto hook = [&]() { ++hooks[tid]; };
      for (int pass = 0; pass < 4; ++pass) {   // as the phases of a launch follow
        c32 x[E];
        __syncthreads();
        for (int i = 0; i < E; ++i) x[i] = in[tf.cb * N + tf.ct + i * T];
        tf.template to_private<false>(x);
        for (int i = 0; i < E; ++i) fwd[tf.pb * N + tf.pt + i * T] = x[i];
        wave_lds_order();   // a wavefront's lanes run together
        if (pass % 2 == 0) {
          tf.template to_coalesced<true>(x, hook);
          for (int i = 0; i < E; ++i) back[tf.cb * N + tf.ct + i * T] = x[i];
        } else {
          tf.spread(x, hook);
          for (int i = 0; i < E; ++i) moved[tf.cb * N + tf.ct + i * T] = x[i];
        }
      }
    });
  for (auto& t : threads) t.join();
  pthread_barrier_destroy(&g_all);
  for (auto& b : g_wave) pthread_barrier_destroy(&b);
  int bad = 0;
  const double e[3] = {error(fwd, re, im), error(back, sre, sim), error(moved, re, im)};
  // FP32 transforms of up to 1024 points, one and two of them
  const double limit = 4e-8 * std::log2((double)N) + 1e-7;
  for (int i = 0; i < 3; ++i)
    if (!(e[i] < 2 * limit)) {
      std::printf("N %d TT %d lean %d: error %d %.3e\n", N, TT, LEAN, i, e[i]);
      ++bad;
    }
  for (int h : hooks) bad += h != 4;
  return bad;
}

template <int N>
int pair_positions() {
  int bad = 0;
  for (int q = 0; q < N / 4; ++q)
    for (int r = 0; r < N; ++r)
      for (int b = 0; b < 2; ++b) {
        const int c = 4 * q + 2 * b;
        bad += 2 * pair_tile_pos<N>(q, b, r) != tpos<2>(N, r, c);
        bad += 2 * pair_tile_pos<N>(q, b, r) + 1 != tpos<2>(N, r, c + 1);
        bad += 2 * pair_mod_pos<N>(q, b, r) != mcb_pos<2>(N, r, c);
        bad += 2 * pair_mod_pos<N>(q, b, r) + 1 != mcb_pos<2>(N, r, c + 1);
        // what the row pass of two rows wrote there, by its thread of 16 values
        constexpr int T = N / 16;
        bad += 2 * pair_dual_pos<N>(q, b, r) != dual_row_pos<N, 2, 16>(r / 2, r % 2, c % T, c / T);
        bad += 2 * pair_dual_pos<N>(q, b, r) + 1 !=
               dual_row_pos<N, 2, 16>(r / 2, r % 2, (c + 1) % T, (c + 1) / T);
      }
  return bad;
}

template <int N, int TT>
int both() { return check<N, TT, false>() + (N <= 512 ? check<N, TT, true>() : 0); }

}  // namespace

int main() {
  const int bad = both<64, 4>() + both<128, 4>() + both<256, 4>() + both<512, 4>() +
                  both<1024, 4>() + both<256, 2>() + both<512, 2>() + pair_positions<2048>() +
                  pair_positions<4096>();
  std::printf("%d bad\n", bad);
  return bad ? 1 : 0;
}
