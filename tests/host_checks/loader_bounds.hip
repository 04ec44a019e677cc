// Host-side check of the direct-to-LDS operand loaders (DldsLoader in gpu_ragged_dot_amd/csrc/rd_gemm_dlds.h), which
// every large-tile core shares - with direct-to-LDS loads and, in the register-staged core, with plain buffer loads.
// No GPU is used: DldsLoader::init / advance are integer arithmetic and run here as they do on the device.
//
// Every K loop in the tree keeps one invariant: the loads of slab s are issued when the loader stands at slab s - advanced
// s times, or, in the streaming routines that begin at a slab of their own, advanced by the first slab's number, then once a
// slab, and back to where it started behind the last one (resource() describes the bytes from slab s to the end of the
// operand window) - with the per-lane offsets
// voff[], and - for a K-major operand whose slab runs past the contraction length - the chunks at or past it replaced
// by an offset beyond the buffer.  Under that invariant this program walks every load of every slab of every wave and
// lane for the loader shapes compiled into the library, on operand windows with ragged edges (row / column limits,
// contraction tails, the DeepSeek-V3 and Mixtral pitches), and checks that
//   * the byte count handed to the buffer resource is positive whenever a load is issued (a count that has gone to zero
//     or below would switch the hardware's range check off);
//   * a load the range check lets through (offset + 16 <= count) reads only elements of the window: row / column below
//     the tile's limit, contraction index below the contraction length and inside the slab being loaded;
//   * every element of the window that belongs to the slab is read exactly once (nothing missing, nothing twice);
//   * every offset is 16-byte aligned and non-negative.
//
// Second part: the loaders of the any-pitch core (RsLoader in gpu_ragged_dot_amd/csrc/rd_gemm_rs.h), whose loads have no
// range check of the hardware behind them.  Same invariant - the loads of slab s are issued with the loader advanced s times,
// here up to kBehind slabs past the last one - on operands that are the whole of their memory: no row in front of the tile's
// first one or behind its last, except what a cut along K leaves on either side.  Every 16-byte piece must lie inside that
// memory, and what trim() and the place in LDS make of it must be, for every row or column below the tile's limit, the
// element of that place, or zero behind the contraction length; every place of a slab is written exactly once.
// Prints "loader_bounds ok <loads checked>" and returns 0, or the first violation and 1.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "rd_gemm_dlds.h"
#include "rd_gemm_rs.h"

using namespace rd;

static long long g_loads = 0;

// start: the slab the walk begins with; past the last slab it goes on with the first.
template <int T, int BK, int NW, bool KMAJOR>
static bool check_window(int lim, int ld, int klen, const char* what, int start = 0) {
  typedef DldsLoader<T, BK, NW, KMAJOR> Ld;
  const int nk = (klen + BK - 1) / BK;
  // all (wave, lane) loaders, advanced in lock step
  std::vector<Ld> ld_all((size_t)NW * 64);
  for (int w = 0; w < NW; ++w)
    for (int l = 0; l < 64; ++l) ld_all[(size_t)w * 64 + l].init(nullptr, ld, lim, klen, w, l);
  const long long window = KMAJOR ? ((long long)(lim - 1) * ld + klen) * 2 : ((long long)(klen - 1) * ld + lim) * 2;
  const std::vector<Ld> first = ld_all;
  if (start > 0)
    for (auto& L : ld_all) L.advance(start);
  std::vector<unsigned char> seen;
  for (int i = 0; i < nk; ++i) {
    const int s = (start + i) % nk;
    const int k0 = s * BK, kend = k0 + BK < klen ? k0 + BK : klen;
    const int rows = KMAJOR ? lim : kend - k0, cols = KMAJOR ? kend - k0 : lim;  // the slab's valid elements, [rows][cols]
    seen.assign((size_t)rows * cols, 0);
    for (int w = 0; w < NW; ++w)
      for (int l = 0; l < 64; ++l) {
        const Ld& L = ld_all[(size_t)w * 64 + l];
        const long long base_bytes = reinterpret_cast<const unsigned char*>(L.base) - static_cast<const unsigned char*>(nullptr);
        if (L.records <= 0) {
          std::printf("%s: T=%d BK=%d NW=%d kmajor=%d lim=%d ld=%d klen=%d slab %d: byte count %d not positive\n", what, T, BK, NW,
                      (int)KMAJOR, lim, ld, klen, s, L.records);
          return false;
        }
        if (base_bytes + L.records != window) {
          std::printf("%s: lim=%d ld=%d klen=%d slab %d: base + count = %lld, window %lld\n", what, lim, ld, klen, s,
                      base_bytes + L.records, window);
          return false;
        }
        const bool tail = k0 + BK > klen;
        for (int j = 0; j < Ld::PER; ++j) {
          int off = L.voff[j];
          if (KMAJOR && tail && k0 + L.kcol >= klen) off = kOobOffset;  // DldsLoader::issue<true>, w4r's fetch_one
          ++g_loads;
          if (off < 0 || (off & 15) != 0) {
            std::printf("%s: lim=%d ld=%d klen=%d slab %d wave %d lane %d load %d: offset %d\n", what, lim, ld, klen, s, w, l, j, off);
            return false;
          }
          if ((long long)off + 16 > L.records) continue;  // out of range: the hardware returns zeros and touches nothing
          const long long e0 = (base_bytes + off) / 2;    // first of 8 elements, from the window's origin
          for (int e = 0; e < 8; ++e) {
            const long long el = e0 + e;
            const long long major = el / ld, minor = el % ld;  // K-major: (row, k); MN-major: (k, column)
            const long long r = KMAJOR ? major : major - k0, c = KMAJOR ? minor - k0 : minor;
            if (r < 0 || r >= rows || c < 0 || c >= cols) {
              std::printf("%s: T=%d BK=%d NW=%d kmajor=%d lim=%d ld=%d klen=%d slab %d wave %d lane %d load %d: element (%lld, %lld) "
                          "outside the slab's %d x %d valid elements\n", what, T, BK, NW, (int)KMAJOR, lim, ld, klen, s, w, l, j, r, c, rows, cols);
              return false;
            }
            if (seen[(size_t)r * cols + c]++) {
              std::printf("%s: lim=%d ld=%d klen=%d slab %d: element (%lld, %lld) read twice\n", what, lim, ld, klen, s, r, c);
              return false;
            }
          }
        }
      }
    for (size_t i = 0; i < seen.size(); ++i)
      if (!seen[i]) {
        std::printf("%s: T=%d BK=%d NW=%d kmajor=%d lim=%d ld=%d klen=%d slab %d: element (%zu, %zu) never read\n", what, T, BK, NW,
                    (int)KMAJOR, lim, ld, klen, s, i / cols, i % cols);
        return false;
      }
    for (size_t l = 0; l < ld_all.size(); ++l) {
      if (s + 1 == nk) ld_all[l].rewind(first[l]);
      else ld_all[l].advance();
    }
  }
  return true;
}

// The streaming routines' walks: from every slab of short contractions - fewer slabs than the ring is deep among them - and from
// the first, second, middle and last of long ones; whole ranges, last slabs that are not full, and pieces of a cut along K.
template <int T, int BK, int NW>
static bool check_rotated(const char* what) {
  for (int ld : {2048, 6144})
    for (int lim : {1, 7, 33, 64, 128, 255, 256})
      for (int klen : {8, 64, 72, 128, 136, 192, 320, 328, 640, 1344, 2048}) {
        if (lim > T) continue;
        const int nk = (klen + BK - 1) / BK;
        for (int start = 0; start < nk; ++start)
          if (nk <= 10 || start < 2 || start == nk / 2 || start == nk - 1)
            if (!check_window<T, BK, NW, true>(lim, ld, klen, what, start)) return false;
      }
  return true;
}

template <int T, int BK, int NW, bool KMAJOR>
static bool check_loader(const char* what) {
  // row pitches: DeepSeek-V3 (2048, 7168), Mixtral (4096, 14336), and small ones; limits and contraction lengths with
  // ragged ends (multiples of 8 where they are row pitches of 16-byte loads: the contraction length of a K-major
  // operand, the column limit of an MN-major one; the rows of a group - tgmm's contraction - are arbitrary)
  const int pitches[] = {2048, 7168, 4096, 14336, 264, T > 256 ? T : 256};
  const int lims_k[] = {1, 4, 7, 21, 33, 64, 100, 128, 129, 255, 256};
  const int lims_mn[] = {8, 24, 64, 120, 128, 136, 248, 256};
  const int klens_k[] = {8, 16, 24, 32, 40, 64, 72, 200, 2040, 2048};
  const int klens_mn[] = {1, 2, 7, 31, 32, 33, 63, 64, 65, 100, 257, 1219};
  for (int ld : pitches)
    for (int lim : (KMAJOR ? std::vector<int>(lims_k, lims_k + 11) : std::vector<int>(lims_mn, lims_mn + 8)))
      for (int klen : (KMAJOR ? std::vector<int>(klens_k, klens_k + 10) : std::vector<int>(klens_mn, klens_mn + 12))) {
        if (lim > T) continue;
        if (KMAJOR ? klen > ld : lim > ld) continue;
        if (!check_window<T, BK, NW, KMAJOR>(lim, ld, klen, what)) return false;
      }
  return true;
}

constexpr int kBehind = 5;  // rs_kloop asks for slab t + 4 in slab t, and an odd number of slabs is rounded up

// A tile at element (0, c0) of a matrix of pitch ld.  K-major: lim rows, contraction indices c0 .. c0 + klen - 1 of each.
// MN-major: klen rows, columns c0 .. c0 + lim - 1 of each.  The memory ends with the matrix's last row.
template <int T, int BK, bool KMAJOR, typename Src, bool VEC, int LB, int NW>
static bool check_rs_window(int lim, int ld, int c0, int klen) {
  typedef RsLoader<T, BK, NW, KMAJOR, Src, VEC, LB> Ld;
  constexpr int EPP = Ld::EPP;
  const int nk = (klen + BK - 1) / BK;
  const long long memory = (long long)(KMAJOR ? lim : klen) * ld;
  const uintptr_t origin = (uintptr_t)1 << 40;
  auto fail = [&](const char* what, int s, int w, int l, int j, long long at) {
    std::printf("any-pitch core: T=%d BK=%d kmajor=%d elem=%d lds=%d vec=%d lim=%d ld=%d c0=%d klen=%d slab %d wave %d lane %d "
                "piece %d: %s (%lld)\n", T, BK, (int)KMAJOR, (int)sizeof(Src), LB, (int)VEC, lim, ld, c0, klen, s, w, l, j, what, at);
    return false;
  };
  std::vector<Ld> all((size_t)NW * 64);
  for (int w = 0; w < NW; ++w)
    for (int l = 0; l < 64; ++l) all[(size_t)w * 64 + l].init(reinterpret_cast<const Src*>(origin) + c0, ld, lim, klen, w, l);
  constexpr int PIECE = EPP * LB;  // bytes of a piece in LDS
  std::vector<unsigned char> placed, written;
  for (int s = 0; s < nk + kBehind; ++s) {
    placed.assign((size_t)(KMAJOR ? T : BK) * Ld::PPR, 0);
    written.assign((size_t)T * BK * LB / PIECE, 0);
    for (int w = 0; w < NW; ++w)
      for (int l = 0; l < 64; ++l) {
        const Ld& L = all[(size_t)w * 64 + l];
        for (int j = 0; j < Ld::PER; ++j) {
          ++g_loads;
          const long long byte = (long long)(reinterpret_cast<uintptr_t>(L.base) - origin) + L.offset(j);
          if (byte % (int)sizeof(Src) != 0) return fail("address inside an element", s, w, l, j, byte);
          const long long first = byte / (int)sizeof(Src);  // of EPP elements, from the matrix's origin
          if (byte < 0 || first + EPP > memory) return fail("load leaves the operand", s, w, l, j, first);
          const int row = Ld::slab_row(w, l, j), piece = l % Ld::PPR;
          if (placed[(size_t)row * Ld::PPR + piece]++) return fail("place taken twice", s, w, l, j, row);
          const int at = L.lds + j * Ld::LDS_STEP;
          if (at < 0 || at % PIECE != 0 || at / PIECE >= (int)written.size() || written[at / PIECE]++)
            return fail("place in LDS", s, w, l, j, at);
          const int down = s >= nk - 1 ? L.surplus(w, l, j, s) : 0;
          if (down < 0) return fail("negative shift", s, w, l, j, down);
          for (int e = 0; e < EPP; ++e) {
            long long got = -1;  // -1: zero
            if (VEC ? down == 0 : e + down < EPP) got = first + e + down;
            const int kk = s * BK + (KMAJOR ? piece * EPP + e : row), mn = KMAJOR ? row : piece * EPP + e;
            if (mn >= lim) continue;
            const long long want = kk >= klen ? -1 : KMAJOR ? (long long)mn * ld + c0 + kk : (long long)kk * ld + c0 + mn;
            if (got != want) return fail("wrong element", s, w, l, j, got);
          }
        }
      }
    for (size_t i = 0; i < placed.size(); ++i)
      if (!placed[i]) return fail("place never written", s, 0, 0, 0, (long long)i);
    for (auto& L : all)
      L.next((int)((&L - all.data()) / 64), (int)((&L - all.data()) % 64));
  }
  return true;
}

template <int T, int BK, bool KMAJOR, typename Src, bool VEC, int LB = 2, int NW = 4>
static bool check_rs_loader() {
  std::vector<int> lims, klens;
  for (int lim : {1, 2, 3, 5, 7, 8, 9, 16, 31, 33, 63, 64, 65, 72, 100, 127, 128, 129, 190, 192, 200, 249, 255, 256})
    if (lim <= T) lims.push_back(lim);
  for (int klen : {1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 24, 31, 32, 33, 40, 57, 63, 64, 65, 72, 95, 96, 97, 127, 128, 129, 136, 191, 192, 193, 200, 257, 333})
    klens.push_back(klen);
  const int widest = (1 << 30) / (512 * (int)sizeof(Src) / 2) - 8;  // 256 rows stay below 2 GiB
  for (int lim : lims)
    for (int klen : klens) {
      if constexpr (KMAJOR) {
        if (VEC && klen % 8 != 0) continue;
        if (klen >= 8 && !check_rs_window<T, BK, true, Src, VEC, LB, NW>(lim, klen, 0, klen)) return false;  // whole rows
        // pieces of a cut along K: they start at multiples of 64 and end at one, or with the row
        for (int c0 : {64, 192})
          for (int behind : {0, 64}) {
            if (behind && klen % 64 != 0) continue;
            if (!check_rs_window<T, BK, true, Src, VEC, LB, NW>(lim, c0 + klen + behind, c0, klen)) return false;
          }
        if (klen % 64 == 0 && (!check_rs_window<T, BK, true, Src, VEC, LB, NW>(lim, klen + 64, 0, klen) ||
                               !check_rs_window<T, BK, true, Src, VEC, LB, NW>(lim, widest, 64, klen))) return false;
      } else {
        if (VEC && lim % 8 != 0) continue;
        // the tile that holds the last columns, of one tile's columns and of several, and one with more behind it
        if (lim >= 8 && !check_rs_window<T, BK, false, Src, VEC, LB, NW>(lim, lim, 0, klen)) return false;
        if (!check_rs_window<T, BK, false, Src, VEC, LB, NW>(lim, T + lim, T, klen)) return false;
        if (lim == T && (!check_rs_window<T, BK, false, Src, VEC, LB, NW>(lim, 2 * T + 24, T, klen) ||
                         !check_rs_window<T, BK, false, Src, VEC, LB, NW>(lim, widest, 0, klen))) return false;
      }
    }
  return true;
}

int main() {
  bool ok = true;
  // (tile extent, slab depth, waves, K-major): the loader shapes of the compiled cores
  ok = ok && check_loader<256, 32, 4, true>("four-wave core, K-major operand");
  ok = ok && check_loader<256, 32, 4, false>("four-wave core, MN-major operand");
  ok = ok && check_loader<256, 64, 4, true>("four-wave register-staged core (64-wide slabs through plain buffer loads)");
  ok = ok && check_loader<256, 32, 8, true>("eight-wave cores, K-major operand");
  ok = ok && check_loader<256, 32, 8, false>("eight-wave cores, MN-major operand");
  ok = ok && check_loader<256, 64, 8, true>("per-operand rings, 64-wide K-major slabs");
  ok = ok && check_loader<128, 32, 8, true>("128 x 256 ping-pong core, rows");
  ok = ok && check_loader<128, 32, 8, false>("128 x 256 ping-pong core, MN-major rows (tgmm)");
  ok = ok && check_loader<128, 32, 4, true>("128 x 128 core, K-major");
  ok = ok && check_loader<128, 32, 4, false>("128 x 128 core, MN-major");
  ok = ok && check_loader<128, 64, 4, false>("128-column tiles, 64-wide MN-major slabs");
  ok = ok && check_loader<256, 64, 4, false>("128 x 256 tiles, 64-wide MN-major slabs");
  ok = ok && check_loader<64, 32, 4, false>("64-column tiles, MN-major") && check_loader<64, 64, 4, false>("64-column tiles, 64-wide MN-major slabs");
  ok = ok && check_loader<64, 32, 4, true>("64-row streaming routine, activations (32-wide slabs)");
  ok = ok && check_loader<64, 64, 4, true>("64-row streaming routine, activations (64-wide slabs)");
  ok = ok && check_loader<128, 64, 4, true>("128-row streaming routine, activations (64-wide slabs)");
  ok = ok && check_rotated<64, 64, 4>("64-row streaming routine from any slab, activations") &&
       check_rotated<128, 64, 4>("128-row streaming routine from any slab, activations") &&
       check_rotated<256, 64, 4>("streaming routines from any slab, weights");
  ok = ok && check_loader<64, 64, 8, true>("eight-wave 64-row routine, activations") && check_loader<128, 64, 8, true>("eight-wave 128-row routine, activations") &&
       check_loader<256, 64, 8, false>("eight-wave short routines, MN-major weights");
  // the any-pitch core's: 16-bit elements, float32 rounded to bf16 at 16-byte pitches and at any, float32 as it is; the row
  // tiles' heights, and the column tiles
  ok = ok && check_rs_loader<64, 64, true, bf16_bits, false>() && check_rs_loader<128, 64, true, bf16_bits, false>() &&
       check_rs_loader<192, 64, true, bf16_bits, false>() && check_rs_loader<256, 64, true, bf16_bits, false>() &&
       check_rs_loader<128, 64, false, bf16_bits, false>() && check_rs_loader<256, 64, false, bf16_bits, false>();
  ok = ok && check_rs_loader<64, 32, true, float, true>() && check_rs_loader<128, 32, true, float, true>() &&
       check_rs_loader<192, 32, true, float, true>() && check_rs_loader<256, 32, true, float, true>() &&
       check_rs_loader<128, 32, false, float, true>() && check_rs_loader<256, 32, false, float, true>();
  ok = ok && check_rs_loader<64, 32, true, float, false>() && check_rs_loader<128, 32, true, float, false>() &&
       check_rs_loader<192, 32, true, float, false>() && check_rs_loader<256, 32, true, float, false>() &&
       check_rs_loader<128, 32, false, float, false>() && check_rs_loader<256, 32, false, float, false>();
  ok = ok && check_rs_loader<64, 32, true, float, false, 4>() && check_rs_loader<128, 32, true, float, false, 4>() &&
       check_rs_loader<64, 32, false, float, false, 4>() && check_rs_loader<128, 32, false, float, false, 4>();
  // the 128 x 256 tile of 16-bit elements, eight waves
  ok = ok && check_rs_loader<64, 64, true, bf16_bits, false, 2, 8>() && check_rs_loader<128, 64, true, bf16_bits, false, 2, 8>() &&
       check_rs_loader<256, 64, true, bf16_bits, false, 2, 8>() && check_rs_loader<128, 64, false, bf16_bits, false, 2, 8>() &&
       check_rs_loader<256, 64, false, bf16_bits, false, 2, 8>();
  // float32 as three bf16 terms on eight waves, and float32 as it is where a tile falls back to it
  ok = ok && check_rs_loader<64, 32, true, float, false, 2, 8>() && check_rs_loader<128, 32, true, float, false, 2, 8>() &&
       check_rs_loader<256, 32, true, float, false, 2, 8>() && check_rs_loader<128, 32, false, float, false, 2, 8>() &&
       check_rs_loader<256, 32, false, float, false, 2, 8>() && check_rs_loader<64, 32, false, float, false, 2>();
  ok = ok && check_rs_loader<192, 32, true, float, false, 2, 8>() && check_rs_loader<64, 32, true, float, true, 2, 8>() &&
       check_rs_loader<128, 32, true, float, true, 2, 8>() && check_rs_loader<192, 32, true, float, true, 2, 8>() &&
       check_rs_loader<256, 32, true, float, true, 2, 8>() && check_rs_loader<256, 32, false, float, true, 2, 8>();
  ok = ok && check_rs_loader<64, 32, true, float, false, 4, 8>() && check_rs_loader<128, 32, true, float, false, 4, 8>() &&
       check_rs_loader<256, 32, true, float, false, 4, 8>() && check_rs_loader<128, 32, false, float, false, 4, 8>() &&
       check_rs_loader<256, 32, false, float, false, 4, 8>();
  if (!ok) return 1;
  std::printf("loader_bounds ok %lld\n", g_loads);
  return 0;
}
