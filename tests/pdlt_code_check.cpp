// Host build of the PDLT v5 decode with code waves (pdlt_host.h, pdlt_lane.h):
// the residual codes by chunk lanes from the chunk table (pdlt_code_chunk)
// into the code buffer, the chains over them in blocks of reconstructions
// alone (pdlt_layout with codes, pdlt_axis_codes), every buffer of exactly
// the launch's size, under the sanitizers when built with them.  Walks,
// triangles and seen counts come from the token lanes (pdlt_tokens).
//
//   pdlt_code_check <stream> <verts.f32 out> <tris.u32 out>
//                   group_size lds_bytes chain32 tok_group staged
//
// staged = 1 reads the codes from the words a code wave stages, 0 from the
// stream itself.  Prints every meshlet's n_int.
// Exit status: 0 ok, 2 stream rejected, 3 no chunk table (a code section past
// its 16-bit positions: the decoder keeps its axis lanes).
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "../meshpress_amd/csrc/pdlt_host.h"

using namespace stride;

template <class T>
static void chains(const PdltHost& H, const std::vector<PdltEntry>& tab,
                   const std::vector<PdltGroup>& groups, uint32_t lds_bytes, const PdltParams& P,
                   const std::vector<uint32_t>& refs, const std::vector<uint32_t>& n_emit,
                   const Walk4* walk, const Walk4* codes, uint64_t cstride, std::vector<float>& V) {
  for (const PdltGroup& G : groups) {
    std::vector<uint64_t> lds((lds_bytes + 7) / 8, 0x5A5A5A5A5A5A5A5Aull);   // stale LDS
    for (uint32_t m = G.m0; m < G.m1; ++m) {
      const PdltEntry& e = tab[m];
      const uint32_t nl = e.n_bnd + e.n_int;
      T* recon = reinterpret_cast<T*>(reinterpret_cast<uint32_t*>(lds.data()) + e.blk_off);
      if (n_emit[m] != e.n_int)
        for (uint32_t i = 0; i < 3 * e.n_int; ++i) recon[(i / e.n_int) * nl + e.n_bnd + i % e.n_int] = 0;
      for (uint32_t i = 0; i < e.n_bnd; ++i)
        for (int d = 0; d < 3; ++d)
          recon[d * nl + i] = (T)pdlt_bnd(H.bnd.at(3ull * refs[e.ref_base + i] + d), P);
      const uint64_t at = pdlt_slot(e.int_base, m, H.n_b);
      for (int d = 0; d < 3; ++d)
        pdlt_axis_codes<T>(e.n_bnd, P, recon + d * nl, walk + at / 4, codes + (d * cstride + at) / 4,
                           n_emit[m]);
      for (uint32_t t = 0; t < 3 * e.n_int; ++t)
        V.at(3ull * e.int_base + t) =
            pdlt_out((double)recon[(t % 3) * nl + e.n_bnd + t / 3], P, (int)(t % 3));
    }
  }
}

int main(int argc, char** argv) {
  if (argc < 9) return 1;
  FILE* f = std::fopen(argv[1], "rb");
  if (!f) return 1;
  std::vector<uint8_t> data;
  uint8_t buf[65536];
  size_t r;
  while ((r = std::fread(buf, 1, sizeof buf, f)) > 0) data.insert(data.end(), buf, buf + r);
  std::fclose(f);
  const bool chain32 = std::atoi(argv[6]) == 1, staged = std::atoi(argv[8]) == 1;
  PdltHost H;
  std::string err;
  if (int rc = pdlt_parse(data.data(), data.size(), H, err)) {
    std::fprintf(stderr, "rejected (%d): %s\n", rc, err.c_str());
    return 2;
  }
  if (H.chunks.empty()) return 3;
  std::vector<PdltEntry> tab = H.tab;
  std::vector<PdltGroup> groups, tg;
  std::vector<ChainEntry> ch;
  std::vector<RefChunk> rch;
  uint32_t lds_bytes = 0, tlds = 0;
  if (pdlt_layout_chains(tab, H.words, 16, std::atoi(argv[7]), tg, ch, rch, tlds, err) ||
      pdlt_layout(tab, std::atoi(argv[4]), std::atoi(argv[5]), groups, lds_bytes, err,
                  chain32 ? 3u : 6u, false, true)) {
    std::fprintf(stderr, "layout: %s\n", err.c_str());
    return 2;
  }
  PdltParams P = H.params;
  P.world = 1;
  P.chain32 = chain32 ? 1 : 0;
  std::vector<float> V(3 * H.n_v);
  std::vector<uint32_t> T(3 * H.n_t), refs(H.n_refs), n_emit(H.n_m);
  for (size_t i = 0; i < H.bnd.size(); ++i) V[i] = pdlt_out(pdlt_bnd(H.bnd[i], P), P, (int)(i % 3));
  // the decoder's buffers (PdltSet::cstride): entries no lane writes stay stale
  const uint64_t cstride = ((uint64_t)(H.n_v - H.n_b) + 4ull * H.n_m + 16 + 3) & ~3ull;
  const Walk4 stale{0x5A5A5A5Au, 0x5A5A5A5Au, 0x5A5A5A5Au, 0x5A5A5A5Au};
  std::vector<Walk4> walk(cstride / 4, stale), codes(3 * cstride / 4, stale);
  for (uint32_t m = 0; m < H.n_m; ++m) {
    const PdltEntry& e = tab[m];
    std::printf("%u\n", e.n_int);
    const uint32_t lo = e.start_bit >> 5, hi = ((e.end_bit - 1) >> 5) + 6;   // read-ahead
    std::vector<uint32_t> st(hi - lo), rl(e.n_bnd), w(e.n_int + 1);
    for (uint32_t i = lo; i < hi; ++i) st[i - lo] = __builtin_bswap32(H.words.at(i));
    std::vector<uint32_t> seen(7 * kTokenSeenStride + 1);
    rl.resize(std::max<uint32_t>(e.n_bnd, 1));   // an interior local's lookup reads refs[0]
    pdlt_tokens<WalkSlot>(st.data(), -32 * (int64_t)lo, e, rl.data(), w.data(),
                          BitSeen{seen.data(), kTokenSeenStride}, &n_emit[m], T.data() + 3ull * e.t_off);
    std::copy(rl.begin(), rl.begin() + e.n_bnd, refs.begin() + e.ref_base);
    uint32_t* slot = reinterpret_cast<uint32_t*>(walk.data()) + pdlt_slot(e.int_base, m, H.n_b);
    for (uint32_t i = 0; i < n_emit[m]; ++i) slot[i] = w[i];
  }
  // the code waves: a lane per 32 walk entries and axis, pieces of four codes
  for (const PdltGroup& G : tg) {
    const uint64_t lo = pdlt_code_lo(tab[G.m0]), n = pdlt_code_words(tab[G.m0], tab[G.m1 - 1]);
    std::vector<uint32_t> st;
    if (staged)
      for (uint64_t i = lo; i < lo + n; ++i) st.push_back(__builtin_bswap32(H.words.at(i)));
    for (uint32_t m = G.m0; m < G.m1; ++m)
      for (uint32_t c = 0; c < (tab[m].n_int + kAxisChunk - 1) / kAxisChunk; ++c)
        for (int d = 0; d < 3; ++d) {
          const PdltEntry& e = tab[m];
          const CodeChunk cc = H.chunks.at((size_t)m * kMaxAxisChunks + c);
          std::vector<uint32_t> row(32, 0x5A5A5A5Au);
          auto out = [&](uint32_t i, uint32_t x) { row.at(i) = x; };
          if (staged) pdlt_code_chunk(LdsStaged{st.data(), lo}, e, cc, c, d, out);
          else pdlt_code_chunk(BufferWords{H.words.data()}, e, cc, c, d, out);
          const uint32_t left = e.n_int - kAxisChunk * c, pieces = (std::min(left, 32u) + 3) / 4;
          const uint64_t at = (d * cstride + pdlt_slot(e.int_base, m, H.n_b)) / 4 + 8u * c;
          for (uint32_t q = 0; q < pieces; ++q)
            codes.at(at + q) = Walk4{row[4 * q], row[4 * q + 1], row[4 * q + 2], row[4 * q + 3]};
        }
  }
  if (chain32)
    chains<float>(H, tab, groups, lds_bytes, P, refs, n_emit, walk.data(), codes.data(), cstride, V);
  else
    chains<double>(H, tab, groups, lds_bytes, P, refs, n_emit, walk.data(), codes.data(), cstride, V);
  FILE* fv = std::fopen(argv[2], "wb");
  FILE* ft = std::fopen(argv[3], "wb");
  if (!fv || !ft) return 1;
  std::fwrite(V.data(), 4, V.size(), fv);
  std::fwrite(T.data(), 4, T.size(), ft);
  std::fclose(fv);
  std::fclose(ft);
  return 0;
}
