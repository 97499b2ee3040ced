// Host build of the residual lanes and code chains of the gfx950 two-pass
// decode (resid_chunk, code_chain in stride_lane.h) against its axis lanes
// (split_axis_g): same codes, from exactly sized buffers.
//
//   resid_check <stream.dpr4>
//
// Prints how many meshlets were compared.  Exit status: 0 ok, 2 stream
// rejected by the pre-pass, 3 codes outside 16 bits (the kernels then keep
// the axis lanes), 4 a code differs.
#include <cstdio>
#include <cstring>
#include <vector>

#include "../meshpress_amd/csrc/stride_lane.h"

using namespace stride;

static uint32_t be32(const uint8_t* p) {
  return ((uint32_t)p[0] << 24) | ((uint32_t)p[1] << 16) | ((uint32_t)p[2] << 8) | p[3];
}

struct Chunks {
  static constexpr bool kOn = true;
  ResidChunk c[kMaxAxisChunks] = {};
  void sub(MeshletScan& s, int j, uint32_t bit) { s.sub_bit[j] = bit; }
  void entry(uint32_t i, uint32_t root) { if (root) c[i >> 5].roots |= 1u << (i & 31u); }
  uint32_t roots(uint32_t i) const { return c[i].roots; }
  void pos(uint32_t i, int s, uint32_t bits) { c[i].pos[s] = (uint16_t)bits; }
};

int main(int argc, char** argv) {
  FILE* f = argc > 1 ? std::fopen(argv[1], "rb") : nullptr;
  if (!f) return 1;
  std::vector<uint8_t> data;
  uint8_t buf[65536];
  size_t r;
  while ((r = std::fread(buf, 1, sizeof buf, f)) > 0) data.insert(data.end(), buf, buf + r);
  std::fclose(f);
  if (data.size() < 86) return 2;
  const uint8_t* d = data.data();
  MeshParams P;
  std::memset(&P, 0, sizeof P);
  for (int i = 0; i < 3; ++i) {
    P.g_bits[i] = d[50 + i];
    P.pred_K[i] = d[71 + i];
  }
  for (int i = 0; i < 9; ++i) P.pred_n[i] = (int16_t)((d[53 + 2 * i] << 8) | d[54 + 2 * i]);
  const uint32_t n_m = be32(d + 82);
  std::vector<uint32_t> le((data.size() + 3) / 4 + 16, 0);   // the device buffer's padding
  std::memcpy(le.data(), d, data.size());
  std::vector<MeshletEntry> tab(n_m);
  std::vector<Chunks> chunks(n_m);
  uint64_t nv = 0;
  for (uint32_t m = 0; m < n_m; ++m) {
    const uint32_t start = be32(d + 86 + 4 * m);
    const uint32_t end = m + 1 < n_m ? be32(d + 86 + 4 * (m + 1)) : (uint32_t)(8 * data.size());
    MeshletScan s, plain;
    GlobalWords src{le.data(), (end + 31u) / 32u + 2u};
    scan_meshlet(src, start, end, P.g_bits, s, chunks[m]);
    scan_meshlet(src, start, end, P.g_bits, plain);   // without the chunk table
    const uint32_t flags = s.flags;
    s.flags &= ~kFlagLongSub;
    if (std::memcmp(&s, &plain, sizeof s)) return 4;
    if (s.error || (flags & kFlagLongSub)) return 2;
    MeshletEntry& e = tab[m];
    e.start_bit = start;
    e.v_off = (uint32_t)nv;
    e.n_local = s.n_local;
    e.n_tris = s.n_tris;
    e.n_strips = s.n_strips | (s.flags & kFlagRawInFifo);
    e.n_kind0 = s.n_kind0;
    e.resid_bit = s.resid_bit;
    for (int j = 0; j < 6; ++j) e.sub_bit[j] = s.sub_bit[j];
    e.end_bit = s.end_bit;
    nv += s.n_local;
  }
  const uint64_t slots = nv + 4ull * n_m + 8, rstride = (slots + 3) & ~3ull;
  std::vector<Walk4> walk4((slots + 3) / 4);
  uint32_t* walk = reinterpret_cast<uint32_t*>(walk4.data());
  std::vector<uint32_t> resid32(3 * rstride / 2, 0xA5A5A5A5u);
  uint16_t* resid = reinterpret_cast<uint16_t*>(resid32.data());
  std::vector<uint32_t> tris(3 * 256 + 9);
  for (uint32_t m = 0; m < n_m; ++m) {
    const MeshletEntry& e = tab[m];
    uint32_t sw[8];
    BitSeen seen{sw};
    seen.preset(0);
    StreamBits cur;
    cur.init(le.data(), e.start_bit + 48);
    split_tokens_c<WalkSlot>(cur, e, walk + walk_slot(P, e, m), seen, tris.data());
    const uint64_t lo = axis_stage_lo(0, e);
    std::vector<uint32_t> ax(axis_stage_words(0, e));
    for (size_t i = 0; i < ax.size(); ++i) ax[i] = __builtin_bswap32(le[lo + i]);
    const LdsStaged staged{ax.data(), lo};
    for (int a = 0; a < 3; ++a) {
      uint16_t* out16 = resid + (uint64_t)a * rstride + walk_slot(P, e, m);
      for (uint32_t c = 0; kAxisChunk * c < e.n_local; ++c) {
        uint32_t left = e.n_local - kAxisChunk * c, n = 0;
        auto out = [&](uint32_t i, uint32_t x) {
          if (i < left) out16[kAxisChunk * c + i] = (uint16_t)x;
          ++n;
        };
        if (axis_rice(staged, 0, e, P, a)) resid_chunk<true>(staged, 0, e, P, chunks[m].c[c], c, a, out);
        else resid_chunk<false>(staged, 0, e, P, chunks[m].c[c], c, a, out);
        if (n != (left < 32 ? left : 32)) return 4;   // every entry once
        // straight from the stream, through the general codeword path
        auto same = [&](uint32_t i, uint32_t x) { n -= out16[kAxisChunk * c + i] == (uint16_t)x; };
        resid_chunk<false>(BufferWords{le.data()}, 0, e, P, chunks[m].c[c], c, a, same);
        if (n) return 4;
      }
    }
  }
  uint32_t compared = 0;
  for (uint32_t m = 0; m < n_m; ++m) {
    const MeshletEntry& e = tab[m];
    const Walk4* wv = reinterpret_cast<const Walk4*>(walk + walk_slot(P, e, m));
    for (int a = 0; a < 3; ++a) {
      if (P.g_bits[a] > 16 || !irlp32_exact(P.pred_n[3 * a], P.pred_n[3 * a + 1], P.pred_n[3 * a + 2], P.pred_K[a]))
        return 3;
      std::vector<uint16_t> want(e.n_local, 0), got(e.n_local, 0x5A5Au);
      if (!split_axis_g<false>(BufferWords{le.data()}, 0, e, P, a, wv, want.data())) return 3;
      CodeChain ch;
      ch.init(P, a);
      code_chain(ch, e.n_local, wv,
                 reinterpret_cast<const uint32_t*>(resid + (uint64_t)a * rstride + walk_slot(P, e, m)),
                 got.data());
      if (want != got) return 4;
    }
    ++compared;
  }
  std::printf("compared %u\n", compared);
  return 0;
}
