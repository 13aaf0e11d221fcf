// C entry points over the tile builder and what a joint step's kernel stages,
// for tests/test_joint_tiles.py (built there with g++).
#include "tiles_shim.cpp"

extern "C" {

// node id that each of a tile's 2 * tile_elems thread-slots stages, and whether
// a joint step reads its u and v from the arrays of the boundary nodes
void tiles_staged(const void* h, int tile, int32_t* id, uint8_t* boundary_row)
{
  const auto* ts = static_cast<const nsm::TileSet*>(h);
  const int   n0 = ts->node_off[(size_t)tile], nn = ts->node_off[(size_t)tile + 1] - n0;
  for (int ln = 0; ln < 2 * ts->tile_elems; ln++) {
    id[ln]           = ts->nodes[(size_t)(n0 + nsm::staged_slot(ln, nn))];
    boundary_row[ln] = nsm::has_boundary_row(id[ln], (int)ts->num_interior);
  }
}
}
