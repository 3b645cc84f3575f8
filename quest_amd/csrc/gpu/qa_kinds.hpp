// The gate kinds of the fusion queue (host planner and device tile code).
#pragma once

namespace qa {
namespace fuse {

// F_DENSEN: an uncontrolled dense matrix on 3 or 4 qubits (a 4-qubit
// superoperator of a density matrix among them), applied to the tile in LDS;
// F_DEPOL2: two-qubit depolarising of a density matrix, its 4 index bits one
// register group; F_DAMP1, F_PAULIS1: damping and the Pauli channel of one qubit;
// F_DEPH2: two-qubit dephasing, diagonal
enum Kind : int {
    F_DENSE1 = 1, F_DENSE2, F_DIAG1, F_PARITY, F_PAULI, F_SWAP, F_DEPOL1, F_DEPH1, F_DENSE1V, F_DENSEN, F_DEPOL2, F_DAMP1,
    F_PAULIS1, F_DEPH2
};

}  // namespace fuse
}  // namespace qa
