// Chip-resident time loop, FDORDER 2, viscoelastic P/SV.
#define DN_F 1
#define DN_GROUP 2
#include "dn_resident_inst.inc"
